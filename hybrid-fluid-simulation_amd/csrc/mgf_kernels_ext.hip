// mgf_kernels_ext.hip — velocity extrapolation of extrapolatingDataInvoker
// (MPhysics/EulerSolverTool.cu:450-557, 904-969).
//
// The reference assigns every face of a component a distance marker by
// breadth-first layers (buildExtrapolationMarkers: layer 0 = known faces,
// layer L = unknown faces with a layer L-1 neighbour, for L < N) and then, for
// L = 1 .. N-1 in order, sets each layer-L face to the mean of its neighbours
// whose marker is below L (extrapolatingData).  The breadth-first search runs
// on the full face grid with no obstacles, so the marker of a face is its L1
// distance to the nearest known face (unknown beyond N-1).  Here:
//
//   1. distance transform, exact and separable: along x the nearest known
//      faces of a row from ballots, along y and z a min-plus transform per
//      line; the z pass also marks the bricks (32 x 16 x 16 faces of one
//      component) that hold a face at distance 1, and the largest distance;
//   2. passes over bricks: a work-group takes a marked brick and its
//      one-face halo into LDS and sets, in layer order, every face whose
//      neighbours one layer below are final; a brick that set a face on one
//      of its sides marks the brick there for the next pass.
//
// The mean is summed in the reference's neighbour order (-x, +x, -y, +y, -z,
// +z) in FP32 and divided once, so the values are bitwise the reference's.
#include <algorithm>
#include <cstring>
#include <vector>

#include "mgf_internal.h"
#include "mgf_kcommon.h"

namespace mgf {

constexpr int32_t kDistInf = 1 << 29;   // unreached (cell distances of the fluid SDF)
// Face distances are stored as uint16 (65535 = unreached): every reachable
// distance is at most nx + ny + nz + 3 < 65535 (the extrapolation refuses
// larger grids), so the transforms compute in int32 and clamp on store.
constexpr int32_t kFaceInf = 0xFFFF;

struct Faces {
    float* f[3];
    uint32_t ex[3], ey[3], ez[3];
    uint32_t off[4];      // first global face index of each component; off[3] = total
    uint32_t rows[4];     // prefix counts of x-rows (ey * ez per component)
    uint32_t ylines[4];   // prefix counts of y-lines (ex * ez)
    uint32_t zlines[4];   // prefix counts of z-lines (ex * ey)
    double rex[3], rexy[3];   // 1/ex, 1/(ex*ey)
};

// Bricks of a component's faces (the unit of a pass, below).
constexpr uint32_t kBrickX = 32, kBrickY = 16, kBrickZ = 16;
__host__ __device__ __forceinline__ uint32_t brick_nx(uint32_t ex) { return (ex + kBrickX - 1) / kBrickX; }
__host__ __device__ __forceinline__ uint32_t brick_ny(uint32_t ey) { return (ey + kBrickY - 1) / kBrickY; }
__host__ __device__ __forceinline__ uint32_t brick_nz(uint32_t ez) { return (ez + kBrickZ - 1) / kBrickZ; }
// First brick of component c (3: all bricks).
__host__ __device__ __forceinline__ uint32_t brick_base(const Faces& F, int c) {
    uint32_t n = 0;
    for (int k = 0; k < 3; ++k)
        if (k < c) n += brick_nx(F.ex[k]) * brick_ny(F.ey[k]) * brick_nz(F.ez[k]);
    return n;
}
// What the z pass of the distance transform leaves for the brick passes:
// mark[brick] = 1 where the brick holds a face at distance 1, and the largest
// distance as the maximum of kFarWords words (spread, so that work-groups do
// not queue at one).
constexpr uint32_t kFarWords = kExtFarWords;
struct ExtSeed {
    uint16_t* mark;
    uint32_t* far;
};

__device__ __forceinline__ int comp_of(const uint32_t (&pre)[4], uint32_t t) {
    return t < pre[1] ? 0 : (t < pre[2] ? 1 : 2);
}

// Per-component values picked with selects: an index into the argument
// arrays with a per-lane component would load them from memory.
template <class T>
__device__ __forceinline__ T pick(const T (&a)[3], int c) {
    return c == 0 ? a[0] : (c == 1 ? a[1] : a[2]);
}
template <class T>
__device__ __forceinline__ T pick4(const T (&a)[4], int c) {
    return c == 0 ? a[0] : (c == 1 ? a[1] : a[2]);
}

__device__ __forceinline__ uint32_t udiv_r(uint32_t a, uint32_t d, double rd) {
    uint32_t q = uint32_t(double(a) * rd);
    const uint32_t r = a - q * d;
    if (int32_t(r) < 0) --q;
    else if (r >= d) ++q;
    return q;
}

// Min-scans over the 64 lanes of a wave: inclusive prefix (lane l gets the
// minimum over lanes 0..l) and suffix (over lanes l..63).  Within each row of
// 16 lanes four DPP row shifts (a lane whose source lies outside its row keeps
// the identity); across the four rows, each row's end lane read with
// v_readlane.  Integer minima, so any order gives the same result.
constexpr int32_t kMinId = 0x7FFFFFFF;
__device__ __forceinline__ int32_t wave_min_prefix(int32_t g) {
    g = min(g, __builtin_amdgcn_update_dpp(kMinId, g, 0x111, 0xF, 0xF, false));   // row_shr:1
    g = min(g, __builtin_amdgcn_update_dpp(kMinId, g, 0x112, 0xF, 0xF, false));   // row_shr:2
    g = min(g, __builtin_amdgcn_update_dpp(kMinId, g, 0x114, 0xF, 0xF, false));   // row_shr:4
    g = min(g, __builtin_amdgcn_update_dpp(kMinId, g, 0x118, 0xF, 0xF, false));   // row_shr:8
    const int32_t r0 = __builtin_amdgcn_readlane(g, 15);
    const int32_t r1 = min(r0, __builtin_amdgcn_readlane(g, 31));
    const int32_t r2 = min(r1, __builtin_amdgcn_readlane(g, 47));
    const uint32_t row = (threadIdx.x & 63) >> 4;
    return min(g, row == 0 ? kMinId : (row == 1 ? r0 : (row == 2 ? r1 : r2)));
}
__device__ __forceinline__ int32_t wave_min_suffix(int32_t h) {
    h = min(h, __builtin_amdgcn_update_dpp(kMinId, h, 0x101, 0xF, 0xF, false));   // row_shl:1
    h = min(h, __builtin_amdgcn_update_dpp(kMinId, h, 0x102, 0xF, 0xF, false));   // row_shl:2
    h = min(h, __builtin_amdgcn_update_dpp(kMinId, h, 0x104, 0xF, 0xF, false));   // row_shl:4
    h = min(h, __builtin_amdgcn_update_dpp(kMinId, h, 0x108, 0xF, 0xF, false));   // row_shl:8
    const int32_t r3 = __builtin_amdgcn_readlane(h, 48);
    const int32_t r2 = min(r3, __builtin_amdgcn_readlane(h, 32));
    const int32_t r1 = min(r2, __builtin_amdgcn_readlane(h, 16));
    const uint32_t row = (threadIdx.x & 63) >> 4;
    return min(h, row == 3 ? kMinId : (row == 2 ? r3 : (row == 1 ? r2 : r1)));
}

// ---------------------------------------------------------------------------
// 1a. Rows along x: d = 0 on known faces, INF elsewhere; then the 1-D L1
// distance: forward d(x) = x + min_{k<=x} (d(k) - k), backward
// d(x) = min_{k>=x} (d(k) + k) - x.  One wave per row.
__device__ __forceinline__ void k_ext_rows_run(Faces F, uint16_t* __restrict__ dist, uint32_t blk, uint32_t slot) {
    (void)blk;
    (void)slot;
    const uint32_t wave = slot * (kBlock / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (wave >= F.rows[3]) return;
    const int c = comp_of(F.rows, wave);
    const uint32_t ex = pick(F.ex, c);
    const uint32_t local = (wave - pick4(F.rows, c)) * ex;     // first face of the row in component c
    const float* f = pick(F.f, c);
    uint16_t* d = dist + pick4(F.off, c) + local;
    // forward
    int32_t carry = kFaceInf;
    for (uint32_t x0 = 0; x0 < ex; x0 += 64) {
        const uint32_t x = x0 + uint32_t(lane);
        const bool ok = x < ex;
        const int32_t d0 = ok ? (f[local + x] != MGF_UNKNOWN ? 0 : kFaceInf) : kFaceInf;
        const int32_t g = min(wave_min_prefix(d0 - int32_t(x)), carry);
        carry = __builtin_amdgcn_readlane(g, 63);
        if (ok) d[x] = uint16_t(min(g + int32_t(x), kFaceInf));
    }
    // backward (each lane re-reads what it wrote)
    carry = 2 * kFaceInf;
    const uint32_t nch = (ex + 63) / 64;
    for (uint32_t ch = nch; ch-- > 0;) {
        const uint32_t x = ch * 64 + uint32_t(lane);
        const bool ok = x < ex;
        const int32_t h = min(wave_min_suffix(ok ? int32_t(d[x]) + int32_t(x) : 2 * kFaceInf), carry);
        carry = __builtin_amdgcn_readlane(h, 0);
        if (ok) d[x] = uint16_t(min(h - int32_t(x), kFaceInf));
    }
}

__global__ void __launch_bounds__(kBlock) k_ext_rows(Faces F, uint16_t* __restrict__ dist) {
    k_ext_rows_run(F, dist, xcd_block(), blockIdx.x);
}

struct MExtRows {
    static constexpr int kThreads = kBlock;
    Faces F;
    uint16_t* dist;
    uint32_t G;
    __device__ void run(uint32_t vb) const { k_ext_rows_run(F, dist, xcd_of(vb, G), vb); }
};

// 1b. Lines along y (axis 1) or z (axis 2): d = min(d, d(prev) + 1) forward
// then backward; one work-item per line, lines x-fastest (coalesced), 32
// loads in flight per chunk (a line is a chain of dependent minima, so the
// loads of a chunk are issued before its first minimum).
template <int AXIS>
__device__ __forceinline__ void k_ext_lines_run(Faces F, uint16_t* __restrict__ dist, ExtSeed seed, uint32_t blk,
                                                uint32_t slot) {
    (void)blk;
    (void)slot;
    const uint32_t t = slot * kBlock + threadIdx.x;
    const uint32_t(&pre)[4] = AXIS == 1 ? F.ylines : F.zlines;
    if (t >= pre[3]) return;
    const int c = comp_of(pre, t);
    const uint32_t l = t - pick4(pre, c);
    const uint32_t ex = pick(F.ex, c), ey = pick(F.ey, c);
    const uint32_t w = udiv_r(l, ex, pick(F.rex, c));
    const uint32_t x = l - w * ex;
    uint32_t start, stride, len;
    if (AXIS == 1) { start = w * ex * ey + x; stride = ex; len = ey; }
    else { start = w * ex + x; stride = ex * ey; len = pick(F.ez, c); }
    uint16_t* d = dist + pick4(F.off, c) + start;
    constexpr int K = 32;
    int32_t prev = kFaceInf;
    for (uint32_t k0 = 0; k0 < len; k0 += K) {
        int32_t v[K];
#pragma unroll
        for (int q = 0; q < K; ++q) v[q] = (k0 + q < len) ? int32_t(d[size_t(k0 + q) * stride]) : 0;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            if (k0 + q < len) {
                prev = min(v[q], prev + 1);
                d[size_t(k0 + q) * stride] = uint16_t(prev);
            }
        }
    }
    prev = kFaceInf;
    uint32_t far = 0;
    const uint32_t nbx = brick_nx(ex), nbxy = nbx * brick_ny(ey);
    uint16_t* mark = AXIS == 2 ? seed.mark + brick_base(F, c) + (w / kBrickY) * nbx + x / kBrickX : nullptr;
    for (uint32_t k1 = len; k1 > 0;) {
        const uint32_t k0 = k1 >= K ? k1 - K : 0;
        const uint32_t m = k1 - k0;
        int32_t v[K];
#pragma unroll
        for (int q = 0; q < K; ++q) v[q] = (uint32_t(q) < m) ? int32_t(d[size_t(k1 - 1 - q) * stride]) : 0;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            if (uint32_t(q) < m) {
                prev = min(v[q], prev + 1);
                d[size_t(k1 - 1 - q) * stride] = uint16_t(min(prev, kFaceInf));
                if (AXIS == 2) {
                    if (prev == 1) mark[((k1 - 1 - q) / kBrickZ) * nbxy] = 1;
                    far = max(far, prev < kFaceInf ? uint32_t(prev) : 0u);
                }
            }
        }
        k1 = k0;
    }
    if (AXIS == 2 && far) atomicMax(&seed.far[t % kFarWords], far);
}

template <int AXIS>
__global__ void __launch_bounds__(kBlock) k_ext_lines(Faces F, uint16_t* __restrict__ dist, ExtSeed seed) {
    k_ext_lines_run<AXIS>(F, dist, seed, xcd_block(), blockIdx.x);
}

template <int AXIS>
struct MExtLines {
    static constexpr int kThreads = kBlock;
    Faces F;
    uint16_t* dist;
    ExtSeed seed;
    uint32_t G;
    __device__ void run(uint32_t vb) const { k_ext_lines_run<AXIS>(F, dist, seed, xcd_of(vb, G), vb); }
};

// 1b'. The same line transform in one read and one write of the distances
// (k_ext_lines re-reads and re-writes them in its backward sweep).  A block of
// kLineSegWaves waves takes 64 consecutive lines (one per lane); wave k holds
// the k-th segment of every line in registers (at most SEG faces).  With
// P_k = min (d(j) - j) and S_k = min (d(j) + j) over segment k, kept in LDS:
//   forward   F(i) = i + min(min_{m<k} P_m, min_{a_k<=j<=i} (d(j) - j))
//   backward  d'(i) = min(min_{m>k} S_m, min_{i<=j<b_k} (F(j) + j)) - i,
// which is min_j (d(j) + |i - j|), the result of the two full-line sweeps
// (integer minima: the same distances).
constexpr int kLineSegWaves = 16;
constexpr int kLineSegThreads = 64 * kLineSegWaves;
constexpr int kLineSegSizes[4] = {12, 20, 36, 64};   // SEG classes: lines of at most 16 SEG faces
constexpr int32_t kSegNone = 1 << 20;                 // past the line's end: above any d(j) +- j

// Stripes of 64 lines in component c (the last one partial).
template <int AXIS>
__device__ __forceinline__ uint32_t seg_stripes(const Faces& F, int c) {
    const uint32_t(&pre)[4] = AXIS == 1 ? F.ylines : F.zlines;
    const uint32_t n = c == 0 ? pre[1] - pre[0] : (c == 1 ? pre[2] - pre[1] : pre[3] - pre[2]);
    return (n + 63) >> 6;
}

template <int AXIS, int SEG, int WAVES = kLineSegWaves>
__device__ __forceinline__ void k_ext_lines_seg_run(Faces F, uint16_t* __restrict__ dist, ExtSeed seed, uint32_t blk,
                                                    uint32_t slot) {
    (void)slot;
    __shared__ int32_t sp[WAVES][64], ss[WAVES][64];
    const uint32_t(&pre)[4] = AXIS == 1 ? F.ylines : F.zlines;
    const uint32_t n0 = seg_stripes<AXIS>(F, 0), n1 = seg_stripes<AXIS>(F, 1), n2 = seg_stripes<AXIS>(F, 2);
    if (blk >= n0 + n1 + n2) return;
    const int c = blk < n0 ? 0 : (blk < n0 + n1 ? 1 : 2);
    const uint32_t sb = blk - (c == 0 ? 0u : (c == 1 ? n0 : n0 + n1));
    const uint32_t lines = c == 0 ? pre[1] - pre[0] : (c == 1 ? pre[2] - pre[1] : pre[3] - pre[2]);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t l = sb * 64 + lane;
    const bool ok = l < lines;
    const uint32_t ex = pick(F.ex, c), ey = pick(F.ey, c);
    const uint32_t w = udiv_r(ok ? l : 0u, ex, pick(F.rex, c));
    const uint32_t x = (ok ? l : 0u) - w * ex;
    uint32_t start, stride, len;
    if (AXIS == 1) { start = w * ex * ey + x; stride = ex; len = ey; }
    else { start = w * ex + x; stride = ex * ey; len = pick(F.ez, c); }
    const uint32_t lb = 2u * (pick4(F.off, c) + start);   // this lane's line start, in bytes (< 2^32)
    const uint32_t seg = (len + WAVES - 1) / WAVES;
    const uint32_t a = wv * seg;
    const uint32_t n = a < len ? min(seg, len - a) : 0u;   // faces of this wave's segment
    uint32_t* far_word = AXIS == 2 ? seed.far + (blk * WAVES + wv) % kFarWords : nullptr;
    const uint32_t seen = AXIS == 2 ? *far_word : 0u;
    // Buffer accesses: the lane's line start in the VGPR offset, the row's
    // wave-uniform byte offset in the SGPR offset (no 64-bit address per row).
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(dist, int16_t(0), int32_t(2u * F.off[3]), kBufWord3);
    const uint32_t rb = 2u * stride;
    int32_t v[SEG];
#pragma unroll
    for (int q = 0; q < SEG; ++q) {
        v[q] = (ok && uint32_t(q) < n) ? int32_t(__builtin_amdgcn_raw_buffer_load_b16(rs, lb, (a + q) * rb, 0))
                                       : kSegNone;
    }
    int32_t pm = kSegNone, sm = kSegNone;
#pragma unroll
    for (int q = 0; q < SEG; ++q) {
        pm = min(pm, v[q] - int32_t(a + q));
        sm = min(sm, v[q] + int32_t(a + q));
    }
    sp[wv][lane] = pm;
    ss[wv][lane] = sm;
    __syncthreads();
    int32_t f = kSegNone, g = kSegNone;
#pragma unroll
    for (int m = 0; m < WAVES; ++m) {
        if (uint32_t(m) < wv) f = min(f, sp[m][lane]);
        if (uint32_t(m) > wv) g = min(g, ss[m][lane]);
    }
#pragma unroll
    for (int q = 0; q < SEG; ++q) {
        f = min(f, v[q] - int32_t(a + q));
        v[q] = f + int32_t(a + q);
    }
#pragma unroll
    for (int q = SEG - 1; q >= 0; --q) {
        g = min(g, v[q] + int32_t(a + q));
        v[q] = g - int32_t(a + q);
    }
    if (AXIS == 2) {
        // the final distances: bricks with a face at distance 1, the largest
        const uint32_t nbx = brick_nx(ex), nbxy = nbx * brick_ny(ey);
        uint16_t* mark = seed.mark + brick_base(F, c) + (w / kBrickY) * nbx + x / kBrickX;
        int32_t far = 0;
        uint32_t hits = 0;   // bit k: a distance of 1 in the k-th brick along z from this segment's first
        const uint32_t za = a / kBrickZ;
#pragma unroll
        for (int q = 0; q < SEG; ++q) {
            if (uint32_t(q) < n) {   // wave-uniform
                hits |= v[q] == 1 ? 1u << ((a + q) / kBrickZ - za) : 0u;
                far = max(far, v[q]);
            }
        }
        // a component is reached everywhere or nowhere
        if (!ok || far >= kFaceInf) far = 0;
        if (!ok) hits = 0;
        far = __builtin_amdgcn_readlane(-wave_min_prefix(-far), 63);
        // one word a wave, spread, and only where it grows (the word as read
        // when the wave began, which may be old)
        if (lane == 0 && uint32_t(far) > seen) atomicMax(far_word, uint32_t(far));
        for (uint32_t k = 0; k <= (SEG + kBrickZ - 1) / kBrickZ; ++k)
            if ((hits >> k) & 1u) mark[(za + k) * nbxy] = 1;
    }
#pragma unroll
    for (int q = 0; q < SEG; ++q) {
        if (ok && uint32_t(q) < n)
            __builtin_amdgcn_raw_buffer_store_b16(uint16_t(min(v[q], kFaceInf)), rs, lb, (a + q) * rb, 0);
    }
}

template <int AXIS, int SEG, int WAVES = kLineSegWaves>
__global__ void __launch_bounds__(64 * WAVES) k_ext_lines_seg(Faces F, uint16_t* __restrict__ dist,
                                                             ExtSeed seed) {
    k_ext_lines_seg_run<AXIS, SEG, WAVES>(F, dist, seed, xcd_block(), blockIdx.x);
}

template <int AXIS, int SEG, int WAVES = kLineSegWaves>
struct MExtLinesSeg {
    static constexpr int kThreads = 64 * WAVES;
    Faces F;
    uint16_t* dist;
    ExtSeed seed;
    uint32_t G;
    __device__ void run(uint32_t vb) const { k_ext_lines_seg_run<AXIS, SEG, WAVES>(F, dist, seed, xcd_of(vb, G), vb); }
};

// Short lines (at most kLineShortWaves * SEG faces) in work-groups of
// kLineShortWaves waves: with 16 waves, a line of 33 faces gives each wave
// 3 faces behind the same loads, exchange and barrier.
constexpr int kLineShortWaves = 4;
constexpr int kLineShortSizes[2] = {12, 36};

// 1a'. The row transform from a ballot of the known faces: a row's
// distances start as 0 (known) or INF, and the two min-plus sweeps of
// k_ext_rows leave at x  min(x - p, n - x, INF), p and n the nearest known
// faces at or before and at or after x (INF where neither exists).  One wave a
// row of at most 64 NCH faces, held in registers; per chunk of 64 faces the
// wave takes the ballot of its known lanes, a lane finds p and n in it with a
// leading- and a trailing-zero count, and the nearest known faces in the
// chunks before and after come from scalar scans of the ballots.  The same
// integers as the sweeps, from one read of the faces and one write of the
// distances.  The faces and distances are raw buffers (the lane's face in a
// 32-bit offset).  At 256^3 this takes 104 us against 125 us for wave-wide
// min-plus scans of the same registers; two, four or eight rows a wave
// measured slower.
template <int NCH>
__device__ __forceinline__ void k_ext_rows_reg_run(Faces F, uint16_t* __restrict__ dist, uint32_t blk, uint32_t slot) {
    (void)blk;
    constexpr int32_t kFar = 1 << 20;   // no known face on that side
    // wave-uniform (readfirstlane), so that the row's component, buffer and
    // bounds live in scalar registers
    const uint32_t row = slot * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    if (row >= F.rows[3]) return;
    const int c = comp_of(F.rows, row);
    const uint32_t ex = pick(F.ex, c);
    const uint32_t local = (row - pick4(F.rows, c)) * ex;
    const uint32_t fb = pick4(F.off, c) + local;   // the row's first face (global index)
    const __amdgpu_buffer_rsrc_t rf = __builtin_amdgcn_make_buffer_rsrc(
        pick(F.f, c), int16_t(0), int32_t(4u * (c == 0 ? F.off[1] - F.off[0] : (c == 1 ? F.off[2] - F.off[1] : F.off[3] - F.off[2]))),
        kBufWord3);
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(dist, int16_t(0), int32_t(2u * F.off[3]), kBufWord3);
    float fv[NCH];
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
        const uint32_t x = uint32_t(ch) * 64 + lane;
        fv[ch] = x < ex ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rf, 4u * (local + x), 0, 0)) : MGF_UNKNOWN;
    }
    uint64_t m[NCH];
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) m[ch] = __ballot(fv[ch] != MGF_UNKNOWN);
    // nearest known faces in the chunks before and after each chunk (scalar)
    int32_t pc[NCH], nc[NCH];
    int32_t run = -kFar;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
        pc[ch] = run;
        if (m[ch]) run = ch * 64 + 63 - __clzll(m[ch]);
    }
    run = kFar;
#pragma unroll
    for (int ch = NCH - 1; ch >= 0; --ch) {
        nc[ch] = run;
        if (m[ch]) run = ch * 64 + __ffsll((unsigned long long)m[ch]) - 1;
    }
    const uint64_t below = (2ull << lane) - 1ull;   // lanes 0 .. lane
    const uint64_t above = ~0ull << lane;            // lanes lane .. 63
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
        const int32_t x = ch * 64 + int32_t(lane);
        if (uint32_t(x) < ex) {
            const uint64_t lo = m[ch] & below, hi = m[ch] & above;
            const int32_t p = lo ? ch * 64 + 63 - __clzll(lo) : pc[ch];
            const int32_t n = hi ? ch * 64 + __ffsll((unsigned long long)hi) - 1 : nc[ch];
            const int32_t d = min(min(x - p, n - x), kFaceInf);
            __builtin_amdgcn_raw_buffer_store_b16(uint16_t(d), rd, 2u * (fb + uint32_t(x)), 0, 0);
        }
    }
}

// Short rows (at most NCH * 64 faces, NCH 1 or 2): the launch is bound by its
// wave count, one wave a row, so a wave takes kRowsPerWave consecutive rows,
// all their loads issued before the first row's distances; each row's
// arithmetic is the one above.
constexpr int kRowsPerWave = 4;

template <int NCH>
__device__ __forceinline__ void k_ext_rows_short_run(Faces F, uint16_t* __restrict__ dist, uint32_t blk,
                                                     uint32_t slot) {
    (void)blk;
    constexpr int32_t kFar = 1 << 20;
    const uint32_t row0 = (slot * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kRowsPerWave;
    const uint32_t lane = threadIdx.x & 63;
    if (row0 >= F.rows[3]) return;
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(dist, int16_t(0), int32_t(2u * F.off[3]), kBufWord3);
    float fv[kRowsPerWave][NCH];
    uint32_t exr[kRowsPerWave], fbr[kRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const uint32_t row = row0 + uint32_t(r);
        const bool ok = row < F.rows[3];
        const int c = comp_of(F.rows, ok ? row : row0);
        const uint32_t ex = ok ? pick(F.ex, c) : 0u;   // a row past the end loads and stores nothing
        const uint32_t local = ok ? (row - pick4(F.rows, c)) * ex : 0u;
        exr[r] = ex;
        fbr[r] = pick4(F.off, c) + local;
        const __amdgpu_buffer_rsrc_t rf = __builtin_amdgcn_make_buffer_rsrc(
            pick(F.f, c), int16_t(0),
            int32_t(4u * (c == 0 ? F.off[1] - F.off[0] : (c == 1 ? F.off[2] - F.off[1] : F.off[3] - F.off[2]))), kBufWord3);
        // loaded unconditionally (past the component's end the buffer reads
        // 0), then the faces past the row replaced
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            const uint32_t x = uint32_t(ch) * 64 + lane;
            const float v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rf, 4u * (local + x), 0, 0));
            fv[r][ch] = x < ex ? v : MGF_UNKNOWN;
        }
    }
    // every row's values in registers before the first row's ballots
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) asm volatile("" : "+v"(fv[r][ch]));
    const uint64_t below = (2ull << lane) - 1ull;   // lanes 0 .. lane
    const uint64_t above = ~0ull << lane;            // lanes lane .. 63
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        uint64_t m[NCH];
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) m[ch] = __ballot(fv[r][ch] != MGF_UNKNOWN);
        int32_t pc[NCH], nc[NCH];
        int32_t run = -kFar;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            pc[ch] = run;
            if (m[ch]) run = ch * 64 + 63 - __clzll(m[ch]);
        }
        run = kFar;
#pragma unroll
        for (int ch = NCH - 1; ch >= 0; --ch) {
            nc[ch] = run;
            if (m[ch]) run = ch * 64 + __ffsll((unsigned long long)m[ch]) - 1;
        }
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            const int32_t x = ch * 64 + int32_t(lane);
            if (uint32_t(x) < exr[r]) {
                const uint64_t lo = m[ch] & below, hi = m[ch] & above;
                const int32_t p = lo ? ch * 64 + 63 - __clzll(lo) : pc[ch];
                const int32_t n = hi ? ch * 64 + __ffsll((unsigned long long)hi) - 1 : nc[ch];
                const int32_t d = min(min(x - p, n - x), kFaceInf);
                __builtin_amdgcn_raw_buffer_store_b16(uint16_t(d), rd, 2u * (fbr[r] + uint32_t(x)), 0, 0);
            }
        }
    }
}

template <int NCH>
__global__ void __launch_bounds__(kBlock) k_ext_rows_short(Faces F, uint16_t* __restrict__ dist) {
    k_ext_rows_short_run<NCH>(F, dist, xcd_block(), blockIdx.x);
}

template <int NCH>
struct MExtRowsShort {
    static constexpr int kThreads = kBlock;
    Faces F;
    uint16_t* dist;
    uint32_t G;
    __device__ void run(uint32_t vb) const { k_ext_rows_short_run<NCH>(F, dist, xcd_of(vb, G), vb); }
};

template <int NCH>
__global__ void __launch_bounds__(kBlock) k_ext_rows_reg(Faces F, uint16_t* __restrict__ dist) {
    k_ext_rows_reg_run<NCH>(F, dist, xcd_block(), blockIdx.x);
}

template <int NCH>
struct MExtRowsReg {
    static constexpr int kThreads = kBlock;
    Faces F;
    uint16_t* dist;
    uint32_t G;
    __device__ void run(uint32_t vb) const { k_ext_rows_reg_run<NCH>(F, dist, xcd_of(vb, G), vb); }
};

// ---------------------------------------------------------------------------
// 2. Passes over bricks.
//
// One launch per layer is bound by launches and latency: a layer is a thin
// shell, 222 of them at 256^3, 8 us each for gathers that move 11x the bytes
// they need, after a counting sort of the faces by distance (0.32 ms); 1.96 ms
// in all (a 256^3 scene whose fluid fills a third of the box).  A brick in LDS
// takes all the layers that cross it in one visit: 18 passes of 74 us there
// (1.34 ms; 512^3: 10.2 -> 4.7 ms).  What bounds a pass is
// a visit's latency, about 20 us (load 5, masks 3, sort 4, a layer 0.3).  Long
// thin grids are chains of passes with one brick or a few each: 65000 x 1 x 1
// faces from one end 55 ms in 2000 passes (by layers 274 ms), 30 x 30 x 2000 6.4
// (6.1), and flat ones fill a sixteenth of a brick: 1000 x 1000 x 1 with a
// thousandth known 1.04 (0.97), from a corner 3.4 (6.2).
//
// Which faces a visit can set: a face at distance L needs its neighbours at
// distance L - 1 (a path down to a known face is a shortest one, so it is
// monotone along each axis), inside the brick or on the halo as the brick was
// loaded.  A face is set (not UNKNOWN) or still UNKNOWN, never anything else: a
// mean over values other than UNKNOWN (FLT_MAX) is FLT_MAX only if its sum
// is, which needs one neighbour that is.  Reading a neighbouring brick's face
// while that brick is being visited gives either, and either is fine: a brick
// that sets a face for which one beyond its side waits marks the brick there
// for the next pass.  By
// induction along the paths, a face is set at the latest in pass
// 1 + (brick sides its longest path crosses), whatever the order of visits, so
// ext_passes() passes set every face, and each face once, from final values.
//
// Marks are stamps: pass p visits the bricks whose stamp in buffer p % 2 is p
// and stamps p + 1 into the other one, so no pass reads what it writes.
// Every work-group counts all stamps of its pass (two bytes a brick, from L2)
// and takes the bricks whose rank is its own index, and every gridDim.x-th
// after it: no list, no counter that all work-groups would queue at.
constexpr int kBrickPer = int(kBrickX) / 4;   // faces a work-item: the 4 x 4 x 4 groups of a wave along x
constexpr int kBrickThreads = int(kBrickX * kBrickY * kBrickZ) / kBrickPer;
constexpr int kHx = int(kBrickX) + 2, kHy = int(kBrickY) + 2, kHz = int(kBrickZ) + 2, kHalo = kHx * kHy * kHz;

struct BrickArgs {
    Faces F;
    const uint16_t* dist;
    int32_t cap;        // layers 1..cap are set
    uint32_t first;     // this scene's first brick among the stamps
};

// LDS of a work-group, 80 KB: two fit a CU.
constexpr int kBrickWaves = kBrickThreads / 64;
constexpr int kBrickFaces = kBrickThreads * kBrickPer;
struct BrickLds {
    float v[kHalo];
    union {
        uint16_t d[kHalo];
        uint32_t list[kBrickFaces];   // by layer: the face's place in v, its mask (m) from bit 14 on
    };
    uint32_t at[kBrickWaves][64];     // a wave's faces by layer
    uint32_t wsum[kBrickWaves];
    int32_t lo, hi;
    uint32_t sides, brick;
};

// One visit; stamps: this scene's bricks in the buffer written.
//
// A layer holds a few of a wave's faces, so a wave that walked its own faces
// layer by layer would run each mean for a few lanes (390 us a pass at 256^3
// that way).  The faces still to be set are first sorted by layer in LDS, and
// a layer's work-items then take list entries densely.  The sort uses no LDS
// atomics (a layer's counter would take them one lane at a time): a wave
// holds 4 x 4 x 4 faces a register, which cross at most 10 layers, finds the
// lanes of one layer with a ballot, and keeps its count of each layer in the
// lane of that number (a brick spans at most 31 + 15 + 15 + 1 layers).
// Bricks of 32 x 8 x 16, 32 x 8 x 8 and 16 x 8 x 8 faces (more passes, more
// stamps) measured slower at 256^3: 8.31, 8.78 and 9.56 ms a step against 8.22.
__device__ __forceinline__ void brick_visit(const BrickArgs& A, uint32_t lb, uint16_t* __restrict__ stamps,
                                            uint32_t pass, BrickLds& S) {
    const Faces& F = A.F;
    int t = threadIdx.x;
    // what depends on the work-item alone is formed in the visit: hoisted out
    // of the loop over bricks it takes the registers of a second work-group
    asm volatile("" : "+v"(t));
    const int lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t b1 = brick_base(F, 1), b2 = brick_base(F, 2);
    const int c = lb < b1 ? 0 : (lb < b2 ? 1 : 2);
    const uint32_t q = lb - (c == 0 ? 0u : (c == 1 ? b1 : b2));
    const int ex = int(pick(F.ex, c)), ey = int(pick(F.ey, c)), ez = int(pick(F.ez, c));
    const uint32_t nbx = brick_nx(ex), nby = brick_ny(ey), nbz = brick_nz(ez);
    const uint32_t bx = q % nbx, by = (q / nbx) % nby, bz = q / (nbx * nby);
    const int x0 = int(bx * kBrickX) - 1, y0 = int(by * kBrickY) - 1, z0 = int(bz * kBrickZ) - 1;
    float* f = pick(F.f, c);
    const uint16_t* dist = A.dist + pick4(F.off, c);
    if (t == 0) {
        S.lo = kFaceInf;
        S.hi = 0;
        S.sides = 0;
    }
    // the brick and its halo; outside the grid: unreached
    constexpr int kLoads = (kHalo + kBrickThreads - 1) / kBrickThreads, kBatch = 11;
#pragma unroll
    for (int k0 = 0; k0 < kLoads; k0 += kBatch) {
        float lv[kBatch];
        uint32_t ld[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int i = (k0 + k) * kBrickThreads + t;
            const int x = x0 + i % kHx, y = y0 + (i / kHx) % kHy, z = z0 + i / (kHx * kHy);
            const bool in = i < kHalo && x >= 0 && y >= 0 && z >= 0 && x < ex && y < ey && z < ez;
            const uint32_t j = in ? (uint32_t(z) * uint32_t(ey) + uint32_t(y)) * uint32_t(ex) + uint32_t(x) : 0u;
            lv[k] = f[j];
            ld[k] = dist[j];
            if (!in) ld[k] = uint32_t(kFaceInf);
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int i = (k0 + k) * kBrickThreads + t;
            if (i < kHalo) {
                S.v[i] = lv[k];
                S.d[i] = uint16_t(ld[k]);
            }
        }
        asm volatile("" ::: "memory");
    }
    __syncthreads();
    // this work-item's faces: the wave's 4 x 4 x 4 groups are k = 0..7 along x
    // in rows of groups along y, then z
    constexpr int kRows = int(kBrickY) / 4;
    const int gy = 4 * (wv % kRows) + ((lane >> 2) & 3), gz = 4 * (wv / kRows) + (lane >> 4);
    const int at0 = ((gz + 1) * kHy + gy + 1) * kHx + (lane & 3) + 1;
    const int nb[6] = {-1, 1, -kHx, kHx, -kHx * kHy, kHx * kHy};
    int32_t d[kBrickPer];
    // neighbours one layer below (0: nothing to set), and from bit 6 on the
    // brick's sides across which a face waits for this one (a face one layer
    // above one still to be set is)
    uint32_t m[kBrickPer];
    int32_t lo = kFaceInf, hi = 0;
    const uint32_t side_yz = (gy == 0 ? 4u : 0u) | (gy == int(kBrickY) - 1 ? 8u : 0u) | (gz == 0 ? 16u : 0u) |
                             (gz == int(kBrickZ) - 1 ? 32u : 0u);
#pragma unroll
    for (int k = 0; k < kBrickPer; ++k) {
        const int o = at0 + 4 * k;
        d[k] = S.d[o];
        int32_t dn[6];
#pragma unroll
        for (int n = 0; n < 6; ++n) dn[n] = S.d[o + nb[n]];
        const bool wait = d[k] >= 1 && d[k] <= A.cap && S.v[o] == MGF_UNKNOWN;
        uint32_t below = 0, above = 0;
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            below |= dn[n] < d[k] ? 1u << n : 0u;
            above |= dn[n] == d[k] + 1 ? 1u << n : 0u;
        }
        const uint32_t side = side_yz | (k == 0 && (lane & 3) == 0 ? 1u : 0u) |
                              (k == kBrickPer - 1 && (lane & 3) == 3 ? 2u : 0u);
        m[k] = wait ? below | ((above & side) << 6) : 0u;
        lo = min(lo, wait ? d[k] : kFaceInf);
        hi = max(hi, wait ? d[k] : 0);
        // two work-groups a CU need 64 VGPRs: not every group's reads at once
        if (k & 1) asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if (lane == 0) {
        atomicMin(&S.lo, lo);
        atomicMax(&S.hi, hi);
    }
    __syncthreads();   // S.d is free from here on
    const int32_t first = __builtin_amdgcn_readfirstlane(S.lo), last = __builtin_amdgcn_readfirstlane(S.hi);
    if (first > last) return;   // nothing to set (the same for every work-item)
    uint32_t rank[kBrickPer], mine = 0;   // mine: the wave's faces of layer first + lane
#pragma unroll
    for (int k = 0; k < kBrickPer; ++k) {
        rank[k] = 0;
        uint64_t todo = __ballot(m[k] != 0);
        while (todo) {
            const int32_t l = __builtin_amdgcn_readlane(d[k], __ffsll((unsigned long long)todo) - 1);
            const uint64_t same = __ballot(m[k] != 0 && d[k] == l);
            const uint32_t had = uint32_t(__builtin_amdgcn_readlane(int(mine), l - first));
            if (d[k] == l) rank[k] = had + __builtin_amdgcn_mbcnt_hi(uint32_t(same >> 32),
                                                                    __builtin_amdgcn_mbcnt_lo(uint32_t(same), 0u));
            if (lane == l - first) mine += uint32_t(__popcll(same));
            todo &= ~same;
        }
    }
    // first list entry of each layer, and of this wave's faces of each: the
    // layer in the lane of its number (every wave for itself)
    S.at[wv][lane] = mine;
    __syncthreads();
    uint32_t all = 0, here = 0;
#pragma unroll
    for (int w = 0; w < kBrickWaves; ++w) {
        const uint32_t x = S.at[w][lane];
        here += w < wv ? x : 0u;
        all += x;
    }
    uint32_t starts = all;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = uint32_t(__shfl_up(int(starts), o, 64));
        if (lane >= o) starts += u;
    }
    const uint32_t faces = uint32_t(__builtin_amdgcn_readlane(int(starts), 63));
    starts -= all;
    here += starts;
#pragma unroll
    for (int k = 0; k < kBrickPer; ++k) {
        const uint32_t to = uint32_t(__shfl(int(here), (m[k] ? d[k] - first : 0), 64)) + rank[k];
        if (m[k]) S.list[to] = uint32_t(at0 + 4 * k) | (m[k] << 14);
    }
    __syncthreads();
    // The layers, one barrier each.  A layer's step is a chain of latencies
    // (list entry, neighbours, sum, quotient, store, barrier), so the next
    // layer's entries are read beside this one's neighbours, waves without an
    // entry skip it, and the sum selects with bit masks.
    const int32_t layers = last - first + 1;
    uint32_t b0 = 0, e0 = uint32_t(__builtin_amdgcn_readlane(int(starts), 1));
    auto entry = [&](uint32_t e) { return S.list[min(e, faces - 1)]; };
    uint32_t next = entry(t);
    auto set = [&](uint32_t e, uint32_t w, uint32_t ahead) {
        const int o = int(w & 0x3FFFu);
        uint32_t fv[6];
#pragma unroll
        for (int n = 0; n < 6; ++n) fv[n] = __float_as_uint(S.v[o + nb[n]]);
        next = entry(ahead);
        // an unused neighbour adds +0: the sum starts at +0, so it is never
        // -0 and stays as it is
        float acc = 0.0f;
        uint32_t known = ~0u;   // 0 once a neighbour used is UNKNOWN
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            const uint32_t u = fv[n] & uint32_t(__builtin_amdgcn_sbfe(int(w), 14 + n, 1));
            known = min(known, u ^ 0x7F7FFFFFu);
            acc += __uint_as_float(u);
        }
        // 1, 2 and 4: the reciprocal and the product are exact as the quotient is
        const uint32_t cnt = uint32_t(__popc((w >> 14) & 63u));
        float mean = acc * __builtin_amdgcn_rcpf(float(cnt));
        if (cnt == 3u || cnt > 4u) mean = acc / float(cnt);
        if (e < e0 && known != 0u) S.v[o] = mean;
    };
    for (int32_t l = 0; l < layers; ++l) {
        const uint32_t b1 = e0, e1 = uint32_t(__builtin_amdgcn_readlane(int(starts), min(l + 2, 63)));
        if (b0 + 64u * uint32_t(wv) < e0) {
            set(b0 + t, next, b1 + t);
            for (uint32_t q = b0 + kBrickThreads; q + 64u * uint32_t(wv) < e0; q += kBrickThreads) set(q + t, entry(q + t), b1 + t);
        } else {
            next = entry(b1 + t);
        }
        b0 = b1;
        e0 = e1;
        __syncthreads();
    }
    // the faces set in this visit, and the sides beyond which one waits for them
    uint32_t sides = 0;
    for (uint32_t e = t; e < faces; e += kBrickThreads) {
        const uint32_t w = S.list[e];
        const int o = int(w & 0x3FFFu);
        const float v = S.v[o];
        if (v != MGF_UNKNOWN) {
            const int lx = o % kHx, ly = (o / kHx) % kHy, lz = o / (kHx * kHy);
            f[(uint32_t(z0 + lz) * uint32_t(ey) + uint32_t(y0 + ly)) * uint32_t(ex) + uint32_t(x0 + lx)] = v;
            sides |= w >> 20;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sides |= uint32_t(__shfl_xor(int(sides), o, 64));
    if (lane == 0 && sides) atomicOr(&S.sides, sides);
    __syncthreads();
    if (t < 6 && ((S.sides >> t) & 1u)) {
        const bool in = t == 0 ? bx > 0 : (t == 1 ? bx + 1 < nbx : (t == 2 ? by > 0 : (t == 3 ? by + 1 < nby
                        : (t == 4 ? bz > 0 : bz + 1 < nbz))));
        const int32_t step = t == 0 ? -1 : (t == 1 ? 1 : (t == 2 ? -int32_t(nbx) : (t == 3 ? int32_t(nbx)
                             : (t == 4 ? -int32_t(nbx * nby) : int32_t(nbx * nby)))));
        if (in) stamps[int64_t(lb) + step] = uint16_t(pass + 1);
    }
    __syncthreads();   // S is reused by the next visit
}

// The bricks of one pass; total: bricks of all scenes, a multiple of 8 with
// padding that is never stamped; scene_of: each brick's scene (null: one).
template <bool MULTI>
__device__ __forceinline__ void bricks_run(const BrickArgs* __restrict__ tab, const BrickArgs& one,
                                           const uint16_t* __restrict__ scene_of, uint16_t* stamps, uint32_t total,
                                           uint32_t pass) {
    __shared__ BrickLds S;
    const uint16_t* rd = stamps + size_t(pass & 1u) * total;
    uint16_t* wr = stamps + size_t((pass + 1u) & 1u) * total;
    const int t = threadIdx.x;
    const uint32_t chunks = total / 8, per = (chunks + kBrickThreads - 1) / kBrickThreads;
    const uint32_t c0 = min(chunks, uint32_t(t) * per), c1 = min(chunks, c0 + per);
    const uint4* rv = reinterpret_cast<const uint4*>(rd);
    auto count = [&](uint32_t w) { return uint32_t((w & 0xFFFFu) == pass) + uint32_t((w >> 16) == pass); };
    uint32_t cnt = 0;
    for (uint32_t i = c0; i < c1; ++i) {
        const uint4 w = rv[i];
        cnt += count(w.x) + count(w.y) + count(w.z) + count(w.w);
    }
    uint32_t incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = uint32_t(__shfl_up(int(incl), o, 64));
        if ((t & 63) >= o) incl += u;
    }
    if ((t & 63) == 63) S.wsum[t >> 6] = incl;
    __syncthreads();
    uint32_t before = incl - cnt, all = 0;
    for (int w = 0; w < kBrickWaves; ++w) {
        if (w < (t >> 6)) before += S.wsum[w];
        all += S.wsum[w];
    }
    for (uint32_t k = blockIdx.x; k < all; k += gridDim.x) {
        if (k >= before && k < before + cnt) {
            uint32_t left = k - before;
            for (uint32_t i = c0 * 8; i < c1 * 8; ++i) {
                if (rd[i] != pass) continue;
                if (left == 0) {
                    S.brick = i;
                    break;
                }
                --left;
            }
        }
        __syncthreads();
        const uint32_t b = S.brick;
        if constexpr (MULTI) {
            const BrickArgs& A = tab[scene_of[b]];
            brick_visit(A, b - A.first, wr + A.first, pass, S);
        } else {
            brick_visit(one, b, wr, pass, S);
        }
    }
}

__global__ void __launch_bounds__(kBrickThreads, 8) k_ext_bricks(BrickArgs A, uint16_t* stamps, uint32_t total,
                                                              uint32_t pass) {
    bricks_run<false>(nullptr, A, nullptr, stamps, total, pass);
}
__global__ void __launch_bounds__(kBrickThreads, 8) k_multi_bricks(const BrickArgs* __restrict__ tab,
                                                                const uint16_t* __restrict__ scene_of,
                                                                uint16_t* stamps, uint32_t total, uint32_t pass) {
    bricks_run<true>(tab, BrickArgs{}, scene_of, stamps, total, pass);
}

// The stamps and the far words, before the distance transform.
__global__ void __launch_bounds__(kBlock) k_ext_zero(uint32_t* __restrict__ a, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) a[i] = 0;
}

// ===========================================================================
// Fields the hybrid coupling reads (GridFluidSolver.cpp:571-613) on the
// cell-centred grid; FluidSurfaceDensity = 0.2 (Common.h:244).

struct Cells {
    uint32_t nx, ny, nz, n;
};

__device__ __forceinline__ void cell_nbrs(const Cells& C, uint32_t i, uint32_t (&j)[6]) {
    const uint32_t sxy = C.nx * C.ny;
    const uint32_t z = i / sxy, rem = i - z * sxy, y = rem / C.nx, x = rem - y * C.nx;
    j[0] = x > 0 ? i - 1 : i;
    j[1] = x + 1 < C.nx ? i + 1 : i;
    j[2] = y > 0 ? i - C.nx : i;
    j[3] = y + 1 < C.ny ? i + C.nx : i;
    j[4] = z > 0 ? i - sxy : i;
    j[5] = z + 1 < C.nz ? i + sxy : i;
}

// buildFluidDensity (MPhysics/EulerSolverTool.cu:408-448): fluid (phi < 0)
// outside the solids (marker >= 0) is 0.2 next to an air cell (phi >= 0 and
// marker >= 0, isInsideAir EulerMathTool.cu:344-348), else 1; the rest 0.
__global__ void __launch_bounds__(kBlock) k_fluid_density(Cells C, const float* __restrict__ phi,
                                                          const float* __restrict__ solid, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= C.n) return;
    uint32_t j[6];
    cell_nbrs(C, i, j);
    bool air = false;
#pragma unroll
    for (int q = 0; q < 6; ++q) air = air || (phi[j[q]] >= 0.0f && solid[j[q]] >= 0.0f);
    const bool fluid = phi[i] < 0.0f && !(solid[i] < 0.0f);
    out[i] = fluid ? (air ? 0.2f : 1.0f) : 0.0f;
}

// buildFluidSDF (MPhysics/EulerSolverTool.cu:324-406) by distance: pass i of
// the reference assigns the cells at breadth-first distance i from the
// boundary layer of their own region (fluid cells with a non-fluid clamped
// neighbour, non-fluid cells with a fluid neighbour).  The nearest boundary
// cell of either region lies in a cell's own region (a path into the other
// region crosses an own boundary cell first), so one L1 distance transform
// from all boundary cells gives both distances.
__global__ void __launch_bounds__(kBlock) k_sdf_seed(Cells C, const float* __restrict__ phi,
                                                     int32_t* __restrict__ d) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= C.n) return;
    uint32_t j[6];
    cell_nbrs(C, i, j);
    const bool in = phi[i] < 0.0f;
    bool other = false;
#pragma unroll
    for (int q = 0; q < 6; ++q) other = other || ((phi[j[q]] < 0.0f) != in);
    d[i] = other ? 0 : kDistInf;
}

// 1-D L1 distance along x rows in place (one wave per row): forward and
// backward min-plus scans as in k_ext_rows.
__global__ void __launch_bounds__(kBlock) k_cdt_rows(Cells C, int32_t* __restrict__ dist) {
    const uint32_t row = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= C.ny * C.nz) return;
    int32_t* d = dist + size_t(row) * C.nx;
    const uint32_t ex = C.nx;
    int32_t carry = kDistInf;
    for (uint32_t x0 = 0; x0 < ex; x0 += 64) {
        const uint32_t x = x0 + uint32_t(lane);
        const bool ok = x < ex;
        const int32_t g = min(wave_min_prefix((ok ? d[x] : kDistInf) - int32_t(x)), carry);
        carry = __builtin_amdgcn_readlane(g, 63);
        if (ok) d[x] = min(g + int32_t(x), kDistInf);
    }
    carry = 2 * kDistInf;
    for (uint32_t ch = (ex + 63) / 64; ch-- > 0;) {
        const uint32_t x = ch * 64 + uint32_t(lane);
        const bool ok = x < ex;
        const int32_t h = min(wave_min_suffix(ok ? d[x] + int32_t(x) : 2 * kDistInf), carry);
        carry = __builtin_amdgcn_readlane(h, 0);
        if (ok) d[x] = min(h - int32_t(x), kDistInf);
    }
}

// Lines along y (AXIS 1) or z (AXIS 2), one work-item per line, x fastest.
template <int AXIS>
__global__ void __launch_bounds__(kBlock) k_cdt_lines(Cells C, int32_t* __restrict__ dist) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t lines = AXIS == 1 ? C.nx * C.nz : C.nx * C.ny;
    if (t >= lines) return;
    const uint32_t w = t / C.nx, x = t - w * C.nx;
    uint32_t start, stride, len;
    if (AXIS == 1) { start = w * C.nx * C.ny + x; stride = C.nx; len = C.ny; }
    else { start = w * C.nx + x; stride = C.nx * C.ny; len = C.nz; }
    int32_t* d = dist + start;
    constexpr int K = 32;
    int32_t prev = kDistInf;
    for (uint32_t k0 = 0; k0 < len; k0 += K) {
        int32_t v[K];
#pragma unroll
        for (int q = 0; q < K; ++q) v[q] = (k0 + q < len) ? d[size_t(k0 + q) * stride] : 0;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            if (k0 + q < len) {
                prev = min(v[q], prev + 1);
                d[size_t(k0 + q) * stride] = prev;
            }
        }
    }
    prev = kDistInf;
    for (uint32_t k1 = len; k1 > 0;) {
        const uint32_t k0 = k1 >= K ? k1 - K : 0;
        const uint32_t m = k1 - k0;
        int32_t v[K];
#pragma unroll
        for (int q = 0; q < K; ++q) v[q] = (uint32_t(q) < m) ? d[size_t(k1 - 1 - q) * stride] : 0;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            if (uint32_t(q) < m) {
                prev = min(v[q], prev + 1);
                d[size_t(k1 - 1 - q) * stride] = min(prev, kDistInf);
            }
        }
        k1 = k0;
    }
}

// Values of buildFluidSDF from the distance d and the region: fluid d = 0 ->
// 0.5-0.2, fluid d -> -(d - (0.5-0.2)), non-fluid d -> d + (1.5-0.2), each
// formed in double and rounded once as the reference's double literals make
// them; d >= passes keeps -UNKNOWN (fluid) or UNKNOWN.
__global__ void __launch_bounds__(kBlock) k_sdf_value(Cells C, const float* __restrict__ phi,
                                                      const int32_t* __restrict__ d, int32_t passes,
                                                      float* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= C.n) return;
    const bool in = phi[i] < 0.0f;
    const int32_t k = d[i];
    float v;
    if (k >= passes) v = in ? -MGF_UNKNOWN : MGF_UNKNOWN;
    else if (in) v = k == 0 ? float(0.5 - 0.2) : float(-(double(k) - (0.5 - 0.2)));
    else v = float(double(k) + (1.5 - 0.2));
    out[i] = v;
}

hipError_t launch_fluid_density(hipStream_t s, const GridDev& g, const float* phi, const float* solid, float* out) {
    const Cells C{uint32_t(g.nx), uint32_t(g.ny), uint32_t(g.nz), uint32_t(g.nx) * g.ny * g.nz};
    (void)launch_dims(k_fluid_density, "k_fluid_density", dim3((C.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, phi, solid, out);
    return hipGetLastError();
}

hipError_t launch_fluid_sdf(hipStream_t s, const GridDev& g, const float* phi, int32_t passes, int32_t* scratch,
                            float* out) {
    const Cells C{uint32_t(g.nx), uint32_t(g.ny), uint32_t(g.nz), uint32_t(g.nx) * g.ny * g.nz};
    const uint32_t G = (C.n + kBlock - 1) / kBlock;
    (void)launch_dims(k_sdf_seed, "k_sdf_seed", dim3(G), dim3(kBlock), 0, s, C, phi, scratch);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    (void)launch_dims(k_cdt_rows, "k_cdt_rows", dim3((C.ny * C.nz + 3) / 4), dim3(kBlock), 0, s, C, scratch);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    (void)launch_dims(k_cdt_lines<1>, "k_cdt_lines", dim3((C.nx * C.nz + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, scratch);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    (void)launch_dims(k_cdt_lines<2>, "k_cdt_lines", dim3((C.nx * C.ny + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, scratch);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    (void)launch_dims(k_sdf_value, "k_sdf_value", dim3(G), dim3(kBlock), 0, s, C, phi, scratch, passes, out);
    return hipGetLastError();
}

// ===========================================================================
static Faces faces_of(const GridDev& g, float* u, float* v, float* w) {
    Faces F;
    F.f[0] = u; F.f[1] = v; F.f[2] = w;
    F.off[0] = F.rows[0] = F.ylines[0] = F.zlines[0] = 0;
    for (int c = 0; c < 3; ++c) {
        F.ex[c] = uint32_t(g.nx + (c == 0));
        F.ey[c] = uint32_t(g.ny + (c == 1));
        F.ez[c] = uint32_t(g.nz + (c == 2));
        F.off[c + 1] = F.off[c] + F.ex[c] * F.ey[c] * F.ez[c];
        F.rows[c + 1] = F.rows[c] + F.ey[c] * F.ez[c];
        F.ylines[c + 1] = F.ylines[c] + F.ex[c] * F.ez[c];
        F.zlines[c + 1] = F.zlines[c] + F.ex[c] * F.ey[c];
        F.rex[c] = 1.0 / double(F.ex[c]);
        F.rexy[c] = 1.0 / (double(F.ex[c]) * double(F.ey[c]));
    }
    return F;
}

int32_t ext_max_distance(const GridDev& g) { return g.nx + g.ny + g.nz + 3; }

// Work-groups of k_ext_rows_reg: a row a wave, 4 waves a group.
static uint32_t rows_grid(const Faces& F, int nch) {
    (void)nch;
    return (F.rows[3] + 3) / 4;
}

// Work-groups of k_ext_rows_short: kRowsPerWave rows a wave, 4 waves a group.
static uint32_t rows_short_grid(const Faces& F) {
    return (F.rows[3] + 4 * kRowsPerWave - 1) / (4 * kRowsPerWave);
}

// The smallest SEG class of k_ext_lines_seg that holds the longest line along
// `axis` (1 = y, 2 = z) in kLineSegWaves segments, or -1 (k_ext_lines then;
// also for 2^31 faces or more, whose byte offsets exceed 32 bits).
static int line_seg_class(const Faces& F, int axis) {
    if (F.off[3] >= (1u << 31)) return -1;
    uint32_t len = 0;
    for (int c = 0; c < 3; ++c) len = std::max(len, axis == 1 ? F.ey[c] : F.ez[c]);
    for (int k = 0; k < 4; ++k)
        if (len <= uint32_t(kLineSegWaves * kLineSegSizes[k])) return k;
    return -1;
}

// The class of k_ext_lines_seg with kLineShortWaves waves for the longest
// line along `axis`, or -1.
static int line_short_class(const Faces& F, int axis) {
    if (F.off[3] >= (1u << 31)) return -1;
    uint32_t len = 0;
    for (int c = 0; c < 3; ++c) len = std::max(len, axis == 1 ? F.ey[c] : F.ez[c]);
    for (int k = 0; k < 2; ++k)
        if (len <= uint32_t(kLineShortWaves * kLineShortSizes[k])) return k;
    return -1;
}

static uint32_t line_seg_grid(const Faces& F, int axis) {
    const uint32_t* pre = axis == 1 ? F.ylines : F.zlines;
    uint32_t n = 0;
    for (int c = 0; c < 3; ++c) n += (pre[c + 1] - pre[c] + 63) / 64;
    return (n + kXcds - 1) / kXcds * kXcds;
}

uint32_t ext_bricks(const GridDev& g) {
    const Faces F = faces_of(g, nullptr, nullptr, nullptr);
    return (brick_base(F, 3) + 7) / 8 * 8;
}

// Passes that set every face within `far` layers: a path of `far` faces
// crosses at most bricks - 1 sides along an axis, and at most one more than
// the brick edges it spans.
uint32_t ext_passes(const GridDev& g, uint32_t far) {
    const Faces F = faces_of(g, nullptr, nullptr, nullptr);
    uint32_t most = 0;
    for (int c = 0; c < 3; ++c) {
        const uint32_t nb[3] = {brick_nx(F.ex[c]), brick_ny(F.ey[c]), brick_nz(F.ez[c])};
        const uint32_t edge[3] = {kBrickX, kBrickY, kBrickZ};
        uint32_t sides = 0, axes = 0, shortest = kBrickX;
        for (int a = 0; a < 3; ++a) {
            sides += nb[a] - 1;
            if (nb[a] > 1) {
                ++axes;
                shortest = std::min(shortest, edge[a]);
            }
        }
        most = std::max(most, std::min(sides, far / shortest + axes));
    }
    return far ? 1 + most : 0;
}

hipError_t launch_ext_zero(hipStream_t s, void* p, size_t words) {
    return launch_dims(k_ext_zero, "k_ext_zero", dim3(uint32_t((words + kBlock - 1) / kBlock)), dim3(kBlock), 0u, s,
                       static_cast<uint32_t*>(p), uint32_t(words));
}

hipError_t launch_ext_distance(hipStream_t s, const GridDev& g, const float* u, const float* v, const float* w,
                               uint16_t* dist, uint16_t* mark, uint32_t* far) {
    const ExtSeed seed{mark, far};
    const Faces F = faces_of(g, const_cast<float*>(u), const_cast<float*>(v), const_cast<float*>(w));
    // rows: held in registers when they fit 16 chunks of 64 faces
    const uint32_t exm = F.ex[0];   // the x-faces have the longest rows
    const double nf = double(F.off[3]);
    probe_next_bytes(6.0 * nf);   // face value 4 read, distance 2 written
    const dim3 b(kBlock);
    if (exm <= 64) (void)launch_dims(k_ext_rows_short<1>, "k_ext_rows_short", dim3(rows_short_grid(F)), b, 0, s, F, dist);
    else if (exm <= 128) (void)launch_dims(k_ext_rows_short<2>, "k_ext_rows_short", dim3(rows_short_grid(F)), b, 0, s, F, dist);
    else if (exm <= 256) (void)launch_dims(k_ext_rows_reg<4>, "k_ext_rows_reg", dim3(rows_grid(F, 4)), b, 0, s, F, dist);
    else if (exm <= 320) (void)launch_dims(k_ext_rows_reg<5>, "k_ext_rows_reg", dim3(rows_grid(F, 5)), b, 0, s, F, dist);
    else if (exm <= 512) (void)launch_dims(k_ext_rows_reg<8>, "k_ext_rows_reg", dim3(rows_grid(F, 8)), b, 0, s, F, dist);
    else if (exm <= 1024) (void)launch_dims(k_ext_rows_reg<16>, "k_ext_rows_reg", dim3(rows_grid(F, 16)), b, 0, s, F, dist);
    else (void)launch_dims(k_ext_rows, "k_ext_rows", dim3((F.rows[3] + 3) / 4), b, 0, s, F, dist);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    for (int axis = 1; axis <= 2; ++axis) {
        probe_next_bytes(4.0 * nf);   // distance 2 read and written
        const int sc = line_short_class(F, axis);
        if (sc >= 0) {
            const dim3 gr(line_seg_grid(F, axis)), bl(64 * kLineShortWaves);
            switch ((axis - 1) * 2 + sc) {
                case 0: (void)launch_dims(k_ext_lines_seg<1, kLineShortSizes[0], kLineShortWaves>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 1: (void)launch_dims(k_ext_lines_seg<1, kLineShortSizes[1], kLineShortWaves>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 2: (void)launch_dims(k_ext_lines_seg<2, kLineShortSizes[0], kLineShortWaves>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                default: (void)launch_dims(k_ext_lines_seg<2, kLineShortSizes[1], kLineShortWaves>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
            }
            const hipError_t e1 = hipGetLastError();
            if (e1 != hipSuccess) return e1;
            continue;
        }
        const int cls = line_seg_class(F, axis);
        if (cls < 0) {
            const uint32_t n = axis == 1 ? F.ylines[3] : F.zlines[3];
            if (axis == 1) (void)launch_dims(k_ext_lines<1>, "k_ext_lines", dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, F, dist, seed);
            else (void)launch_dims(k_ext_lines<2>, "k_ext_lines", dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, F, dist, seed);
        } else {
            const dim3 gr(line_seg_grid(F, axis)), bl(kLineSegThreads);
            switch ((axis - 1) * 4 + cls) {
                case 0: (void)launch_dims(k_ext_lines_seg<1, kLineSegSizes[0]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 1: (void)launch_dims(k_ext_lines_seg<1, kLineSegSizes[1]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 2: (void)launch_dims(k_ext_lines_seg<1, kLineSegSizes[2]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 3: (void)launch_dims(k_ext_lines_seg<1, kLineSegSizes[3]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 4: (void)launch_dims(k_ext_lines_seg<2, kLineSegSizes[0]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 5: (void)launch_dims(k_ext_lines_seg<2, kLineSegSizes[1]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                case 6: (void)launch_dims(k_ext_lines_seg<2, kLineSegSizes[2]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
                default: (void)launch_dims(k_ext_lines_seg<2, kLineSegSizes[3]>, "k_ext_lines_seg", gr, bl, 0, s, F, dist, seed); break;
            }
        }
        const hipError_t e2 = hipGetLastError();
        if (e2 != hipSuccess) return e2;
    }
    return hipSuccess;
}

// Work-groups of a pass: two fit each of 256 CUs; each takes every 512th brick.
constexpr uint32_t kBrickGroups = 512;

hipError_t launch_ext_bricks(hipStream_t s, const GridDev& g, float* u, float* v, float* w, const uint16_t* dist,
                             int32_t cap, uint16_t* stamps, uint32_t pass) {
    const uint32_t total = ext_bricks(g);
    const BrickArgs A{faces_of(g, u, v, w), dist, cap, 0u};
    return launch_dims(k_ext_bricks, "k_ext_bricks", dim3(std::min(total, kBrickGroups)), dim3(kBrickThreads), 0u, s, A,
                       stamps, total, pass);
}

// ===========================================================================
// Multi-scene records of the distance transform (launch_ext_distance): the
// same arguments and grids.
template <class A>
static void push_rec_e(std::vector<MRec>& out, int32_t kind, const A& a, uint32_t blocks) {
    static_assert(sizeof(A) <= kMRecBytes, "argument struct fits a record");
    MRec r;
    r.kind = kind;
    r.blocks = blocks;
    r.bytes = uint32_t(sizeof(A));
    std::memcpy(r.args, &a, sizeof(A));
    out.push_back(r);
}

void rec_ext_distance(std::vector<MRec>& out, const GridDev& g, float* u, float* v, float* w, uint16_t* dist,
                      uint16_t* mark, uint32_t* far) {
    const ExtSeed seed{mark, far};
    const Faces F = faces_of(g, u, v, w);
    const uint32_t exm = F.ex[0];
    const uint32_t rg = (F.rows[3] + 3) / 4;
    if (exm <= 64) push_rec_e(out, kMkExtRowsShort1, MExtRowsShort<1>{F, dist, rows_short_grid(F)}, rows_short_grid(F));
    else if (exm <= 128) push_rec_e(out, kMkExtRowsShort2, MExtRowsShort<2>{F, dist, rows_short_grid(F)}, rows_short_grid(F));
    else if (exm <= 256) push_rec_e(out, kMkExtRowsReg4, MExtRowsReg<4>{F, dist, rows_grid(F, 4)}, rows_grid(F, 4));
    else if (exm <= 320) push_rec_e(out, kMkExtRowsReg5, MExtRowsReg<5>{F, dist, rows_grid(F, 5)}, rows_grid(F, 5));
    else if (exm <= 512) push_rec_e(out, kMkExtRowsReg8, MExtRowsReg<8>{F, dist, rows_grid(F, 8)}, rows_grid(F, 8));
    else if (exm <= 1024) push_rec_e(out, kMkExtRowsReg16, MExtRowsReg<16>{F, dist, rows_grid(F, 16)}, rows_grid(F, 16));
    else push_rec_e(out, kMkExtRows, MExtRows{F, dist, rg}, rg);
    for (int axis = 1; axis <= 2; ++axis) {
        const int sc = line_short_class(F, axis);
        if (sc >= 0) {
            const uint32_t gl = line_seg_grid(F, axis);
            const int32_t kind = kMkExtLinesShort + (axis - 1) * 2 + sc;
            switch ((axis - 1) * 2 + sc) {
                case 0: push_rec_e(out, kind, MExtLinesSeg<1, kLineShortSizes[0], kLineShortWaves>{F, dist, seed, gl}, gl); break;
                case 1: push_rec_e(out, kind, MExtLinesSeg<1, kLineShortSizes[1], kLineShortWaves>{F, dist, seed, gl}, gl); break;
                case 2: push_rec_e(out, kind, MExtLinesSeg<2, kLineShortSizes[0], kLineShortWaves>{F, dist, seed, gl}, gl); break;
                default: push_rec_e(out, kind, MExtLinesSeg<2, kLineShortSizes[1], kLineShortWaves>{F, dist, seed, gl}, gl); break;
            }
            continue;
        }
        const int cls = line_seg_class(F, axis);
        if (cls < 0) {
            const uint32_t gl = ((axis == 1 ? F.ylines[3] : F.zlines[3]) + kBlock - 1) / kBlock;
            if (axis == 1) push_rec_e(out, kMkExtLines1, MExtLines<1>{F, dist, seed, gl}, gl);
            else push_rec_e(out, kMkExtLines2, MExtLines<2>{F, dist, seed, gl}, gl);
            continue;
        }
        const uint32_t gl = line_seg_grid(F, axis);
        const int32_t kind = kMkExtLinesSeg + (axis - 1) * 4 + cls;
        switch ((axis - 1) * 4 + cls) {
            case 0: push_rec_e(out, kind, MExtLinesSeg<1, kLineSegSizes[0]>{F, dist, seed, gl}, gl); break;
            case 1: push_rec_e(out, kind, MExtLinesSeg<1, kLineSegSizes[1]>{F, dist, seed, gl}, gl); break;
            case 2: push_rec_e(out, kind, MExtLinesSeg<1, kLineSegSizes[2]>{F, dist, seed, gl}, gl); break;
            case 3: push_rec_e(out, kind, MExtLinesSeg<1, kLineSegSizes[3]>{F, dist, seed, gl}, gl); break;
            case 4: push_rec_e(out, kind, MExtLinesSeg<2, kLineSegSizes[0]>{F, dist, seed, gl}, gl); break;
            case 5: push_rec_e(out, kind, MExtLinesSeg<2, kLineSegSizes[1]>{F, dist, seed, gl}, gl); break;
            case 6: push_rec_e(out, kind, MExtLinesSeg<2, kLineSegSizes[2]>{F, dist, seed, gl}, gl); break;
            default: push_rec_e(out, kind, MExtLinesSeg<2, kLineSegSizes[3]>{F, dist, seed, gl}, gl); break;
        }
    }
}

size_t brick_arg_bytes() { return sizeof(BrickArgs); }

void brick_args(unsigned char* dst, const GridDev& g, float* u, float* v, float* w, const uint16_t* dist, int32_t cap,
                uint32_t first) {
    const BrickArgs a{faces_of(g, u, v, w), dist, cap, first};
    std::memcpy(dst, &a, sizeof(BrickArgs));
}

hipError_t launch_multi_bricks(hipStream_t s, const void* tab, const uint16_t* scene_of, uint16_t* stamps,
                               uint32_t total, uint32_t pass) {
    return launch_dims(k_multi_bricks, "k_multi_bricks", dim3(std::min(total, kBrickGroups)), dim3(kBrickThreads), 0u, s,
                       static_cast<const BrickArgs*>(tab), scene_of, stamps, total, pass);
}

template <class A>
static hipError_t launch_me(hipStream_t s, const char* name, const void* tab, const uint32_t* map, uint32_t nblocks,
                            const uint8_t* active) {
    return launch_dims(k_multi<A>, name, dim3(nblocks), dim3(A::kThreads), 0u, s, static_cast<const A*>(tab), map,
                       active);
}

hipError_t launch_multi_ext(hipStream_t s, int32_t kind, const void* tab, const uint32_t* map, uint32_t nblocks,
                            uint32_t, const uint8_t* active) {
    switch (kind) {
        case kMkExtRows: return launch_me<MExtRows>(s, "k_multi_ext_rows", tab, map, nblocks, active);
        case kMkExtLinesShort + 0: return launch_me<MExtLinesSeg<1, kLineShortSizes[0], kLineShortWaves>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesShort + 1: return launch_me<MExtLinesSeg<1, kLineShortSizes[1], kLineShortWaves>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesShort + 2: return launch_me<MExtLinesSeg<2, kLineShortSizes[0], kLineShortWaves>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesShort + 3: return launch_me<MExtLinesSeg<2, kLineShortSizes[1], kLineShortWaves>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtRowsShort1: return launch_me<MExtRowsShort<1>>(s, "k_multi_ext_rows_short", tab, map, nblocks, active);
        case kMkExtRowsShort2: return launch_me<MExtRowsShort<2>>(s, "k_multi_ext_rows_short", tab, map, nblocks, active);
        case kMkExtRowsReg4: return launch_me<MExtRowsReg<4>>(s, "k_multi_ext_rows_reg", tab, map, nblocks, active);
        case kMkExtRowsReg5: return launch_me<MExtRowsReg<5>>(s, "k_multi_ext_rows_reg", tab, map, nblocks, active);
        case kMkExtRowsReg8: return launch_me<MExtRowsReg<8>>(s, "k_multi_ext_rows_reg", tab, map, nblocks, active);
        case kMkExtRowsReg16: return launch_me<MExtRowsReg<16>>(s, "k_multi_ext_rows_reg", tab, map, nblocks, active);
        case kMkExtLines1: return launch_me<MExtLines<1>>(s, "k_multi_ext_lines", tab, map, nblocks, active);
        case kMkExtLines2: return launch_me<MExtLines<2>>(s, "k_multi_ext_lines", tab, map, nblocks, active);
        case kMkExtLinesSeg + 0: return launch_me<MExtLinesSeg<1, kLineSegSizes[0]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 1: return launch_me<MExtLinesSeg<1, kLineSegSizes[1]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 2: return launch_me<MExtLinesSeg<1, kLineSegSizes[2]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 3: return launch_me<MExtLinesSeg<1, kLineSegSizes[3]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 4: return launch_me<MExtLinesSeg<2, kLineSegSizes[0]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 5: return launch_me<MExtLinesSeg<2, kLineSegSizes[1]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 6: return launch_me<MExtLinesSeg<2, kLineSegSizes[2]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        case kMkExtLinesSeg + 7: return launch_me<MExtLinesSeg<2, kLineSegSizes[3]>>(s, "k_multi_ext_lines_seg", tab, map, nblocks, active);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mgf
