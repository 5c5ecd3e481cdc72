// mgf_kernels_particles.hip — particle <-> grid transfers and particle
// advection of CEulerParticles (MPhysics/EulerParticles.cpp,
// MPhysics/EulerParticlesTool.cu), the primitives of the PIC / FLIP / mixed
// advection solvers (MPhysics/ParticleInCell.cpp, FluidImplicitParticle.cpp,
// MixPICAndFLIP.cpp).
//
// Particle positions and per-particle vectors are interleaved x, y, z
// (3 * i + k), as the reference stores them.  One work-item per particle,
// where nothing else is said.  Particle-to-grid sums have no fixed order, as the
// reference's FP32 atomics have none: the tile-sorted splat sums a cell's
// particles in the order in which they were ranked in LDS, and adds every node
// that a tile's particles touch to the fields by atomics (two a node, one for
// P2GSUM, which has no weight); the unsorted one adds to LDS by atomics too.
// Grid-to-particle sums, counts and the advection are order-free and bitwise
// the oracle's.
#include "mgf_internal.h"
#include "mgf_kcommon.h"

namespace mgf {

// A cell-centred grid of extents n, origin o, spacing h: a field of cells, or
// one component of a face-centred field (its extents and origin shifted by
// -h/2 on its axis).
struct PGrid {
    int nx, ny, nz;
    float ox, oy, oz, hx, hy, hz;
    float rhx, rhy, rhz;   // 1/h, used when every spacing is a power of two (pow2)
    int pow2;
};

// Transfer kernels (MPhysics/EulerMathTool.cu:268-294): written with double
// literals in the reference, so evaluated in double from the float argument
// and rounded once.
__device__ __forceinline__ float pg_linear(float v) {
    const float a = fabsf(v);
    return a < 1.0f ? float(1.0 - double(a)) : 0.0f;
}
__device__ __forceinline__ float pg_quadratic(float v) {
    const float a = fabsf(v);
    if (a < 0.5f) return float(0.75 - double(a * a));
    if (a < 1.5f) return float(0.5 * (1.5 - double(a)) * (1.5 - double(a)));
    return 0.0f;
}
__device__ __forceinline__ float pg_cubic(float v) {
    const float a = fabsf(v);
    if (a < 1.0f) return float(0.5 * double(a) * double(a) * double(a) - double(a * a) + 2.0 / 3.0);
    if (a < 2.0f) return float(1.0 / 6.0 * (2.0 - double(a)) * (2.0 - double(a)) * (2.0 - double(a)));
    return 0.0f;
}

// transPos2Index (EulerMathTool.cu:29-40): truncation of (p - o) / h, clamped.
__device__ __forceinline__ uint32_t pos_cell(const PGrid& g, float px, float py, float pz) {
    const int ix = clampi(int(div_h(px - g.ox, g.hx, g.rhx, g.pow2)), g.nx);
    const int iy = clampi(int(div_h(py - g.oy, g.hy, g.rhy, g.pow2)), g.ny);
    const int iz = clampi(int(div_h(pz - g.oz, g.hz, g.rhz, g.pow2)), g.nz);
    return (uint32_t(iz) * uint32_t(g.ny) + uint32_t(iy)) * uint32_t(g.nx) + uint32_t(ix);
}

// The support of a particle (EulerParticlesTool.cu:97-101, 216-220): lower
// corner and per-axis weights; n = 2 (linear) or 4 (corners i0-1 .. i0+2).
struct PStencil {
    int i0[3];
    float w[3][4];
};
// One axis of the support: lower corner and the kernel's weights.
__device__ __forceinline__ void pg_axis(float rel, float h, float rh, int pow2, int alg, int& i0, float (&w)[4]) {
    i0 = floor_ref(div_h(rel, h, rh, pow2));
    const float f = div_h(rel - float(i0) * h, h, rh, pow2);
    if (alg == MGF_PG_LINEAR) {
        w[0] = pg_linear(f);
        w[1] = pg_linear(float(double(f) - 1.0));
        w[2] = w[3] = 0.0f;
    } else if (alg == MGF_PG_QUADRATIC) {
        w[0] = pg_quadratic(float(double(f) + 1.0));
        w[1] = pg_quadratic(float(double(f) + 1.0 - 1.0));
        w[2] = pg_quadratic(float(double(f) + 1.0 - 2.0));
        w[3] = pg_quadratic(float(double(f) + 1.0 - 3.0));
    } else {
        w[0] = pg_cubic(float(double(f) + 1.0));
        w[1] = pg_cubic(float(double(f) + 1.0 - 1.0));
        w[2] = pg_cubic(float(double(f) + 1.0 - 2.0));
        w[3] = pg_cubic(float(double(f) + 1.0 - 3.0));
    }
}

__device__ __forceinline__ void pg_stencil(const PGrid& g, float px, float py, float pz, int alg, PStencil& st) {
    pg_axis(px - g.ox - g.hx * 0.5f, g.hx, g.rhx, g.pow2, alg, st.i0[0], st.w[0]);
    pg_axis(py - g.oy - g.hy * 0.5f, g.hy, g.rhy, g.pow2, alg, st.i0[1], st.w[1]);
    pg_axis(pz - g.oz - g.hz * 0.5f, g.hz, g.rhz, g.pow2, alg, st.i0[2], st.w[2]);
}

__device__ __forceinline__ uint32_t pg_index(const PGrid& g, int x, int y, int z) {
    return lin3(x, y, z, g.nx, g.ny, g.nz);
}

// The corners of a support in the reference's order (z, y, x), with their
// weights w_x * w_y * w_z; N = 2 (LINEAR, corners i0 .. i0+1) or 4
// (QUADRATIC / CUBIC, corners i0-1 .. i0+2), unrolled so the weights stay in
// registers.
template <int N, class F>
__device__ __forceinline__ void for_corners(const PGrid& g, const PStencil& st, F&& f) {
    constexpr int lo = N == 2 ? 0 : -1;
#pragma unroll
    for (int z = 0; z < N; ++z)
#pragma unroll
        for (int y = 0; y < N; ++y)
#pragma unroll
            for (int x = 0; x < N; ++x)
                f(pg_index(g, st.i0[0] + x + lo, st.i0[1] + y + lo, st.i0[2] + z + lo),
                  st.w[0][x] * st.w[1][y] * st.w[2][z]);
}

// The splat over particles in any order (the operator, and the solvers' wide
// kernels).  What bounds it is where a corner's sum lands: QUADRATIC adds 27
// and CUBIC 64 values and weights a particle, and an FP32 atomic costs about
// five cycles a lane in LDS and far more in global memory.  So no corner is
// added with an atomic: the particles are sorted by the 8^3-cell tile of their
// lowest corner (k_splat_count, k_splat_scan, k_splat_order), and a work-group
// takes up to kSplatChunk particles of one tile, sorts them by cell in LDS,
// sums each cell's particles in the registers of one work-item (a slot per
// corner) and adds the slots to a dense LDS tile of nodes one corner at a
// time: for a fixed corner the cells' nodes are distinct, so plain adds do.
// The tile is flushed with global atomics, one a field and node touched.
// 1.23M QUADRATIC particles on 101 x 83 x 61 cells, one field: 10.0 ms with an
// LDS hash table of a work-group's nodes, 0.54 ms (after the same sort) with
// LDS float atomics per corner, 0.081 ms this way (and 0.035 ms for the sort).
constexpr int kTileEdge = 8;
constexpr int kSplatBlock = kTileEdge * kTileEdge * kTileEdge;   // a work-item a cell
constexpr uint32_t kSplatRounds = 4;
constexpr uint32_t kSplatChunk = kSplatRounds * kSplatBlock;
// Particles of a cell summed by its own work-item; what a denser cell holds
// beyond is summed by all work-items, kSplatRounds each.
constexpr uint32_t kSplatCell = 64;
// Particles sorted at a time: bounds the scratch; the sums just continue.
constexpr int64_t kSplatSegment = int64_t(1) << 24;
// A work-group of the sort counts its particles through LDS in a window of this
// many tiles (32 KB) around the tile of one of them: all tiles of a grid of up
// to 160^3 cells; beyond, the tiles of the particles' neighbourhood, since sets
// are generated cell by cell and move little against their order.  Particles
// outside the window take global atomics, one a tile and wave.
constexpr uint32_t kSplatLdsTiles = 8192;
constexpr uint32_t kSplatItems = 16;                             // particles a work-item of those passes

// Corners an axis with a weight: QUADRATIC has three of its four (the outer
// one at least 1.5 away is +0).
constexpr int splat_corners(int alg) {
    return alg == MGF_PG_P2GSUM ? 1 : (alg == MGF_PG_LINEAR ? 2 : (alg == MGF_PG_QUADRATIC ? 3 : 4));
}

// Tiles an axis of n nodes: the lowest corner is clamped to [-(N - 1), n - 1]
// (corners clamp to the grid, so a support further out covers the same nodes).
__host__ __device__ __forceinline__ uint32_t splat_tiles(int n, int N) {
    return uint32_t(n + N - 1 + kTileEdge - 1) / uint32_t(kTileEdge);
}

// One axis: the lowest corner with a weight, not clamped (P2GSUM: the cell).
template <int ALG>
__device__ __forceinline__ int splat_first(float p, float o, float h, float rh, int pow2, int n) {
    if constexpr (ALG == MGF_PG_P2GSUM) return clampi(int(div_h(p - o, h, rh, pow2)), n);
    const float rel = p - o - h * 0.5f;
    const int b = floor_ref(div_h(rel, h, rh, pow2));
    if constexpr (ALG == MGF_PG_LINEAR) return b;
    if constexpr (ALG == MGF_PG_CUBIC) return b - 1;
    const float f = div_h(rel - float(b) * h, h, rh, pow2);
    return fabsf(float(double(f) + 1.0)) < 1.5f ? b - 1 : b;   // pg_quadratic of it is not 0
}

// Clamped and shifted to start at 0.
template <int ALG>
__device__ __forceinline__ int splat_low(float p, float o, float h, float rh, int pow2, int n) {
    constexpr int N = splat_corners(ALG);
    const int b = splat_first<ALG>(p, o, h, rh, pow2, n);
    return (b < -(N - 1) ? -(N - 1) : (b > n - 1 ? n - 1 : b)) + N - 1;
}

struct SplatAt {
    uint32_t tile, cell;
};
template <int ALG>
__device__ __forceinline__ SplatAt splat_at(const PGrid& g, float px, float py, float pz) {
    constexpr int N = splat_corners(ALG);
    const uint32_t x = uint32_t(splat_low<ALG>(px, g.ox, g.hx, g.rhx, g.pow2, g.nx));
    const uint32_t y = uint32_t(splat_low<ALG>(py, g.oy, g.hy, g.rhy, g.pow2, g.ny));
    const uint32_t z = uint32_t(splat_low<ALG>(pz, g.oz, g.hz, g.rhz, g.pow2, g.nz));
    SplatAt a;
    a.tile = ((z / kTileEdge) * splat_tiles(g.ny, N) + y / kTileEdge) * splat_tiles(g.nx, N) + x / kTileEdge;
    a.cell = ((z % kTileEdge) * kTileEdge + y % kTileEdge) * kTileEdge + x % kTileEdge;
    return a;
}
template <int ALG>
__device__ __forceinline__ SplatAt splat_at(const PGrid& g, const float* __restrict__ pos, size_t p) {
    return splat_at<ALG>(g, pos[3 * p], pos[3 * p + 1], pos[3 * p + 2]);
}

// Zeros for the field and the weight (first segment) and the tile counters.
__global__ void __launch_bounds__(kBlock) k_splat_clear(size_t n, float* __restrict__ field, float* __restrict__ weight,
                                                        size_t nt, uint32_t* __restrict__ counts) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n) {
        field[i] = 0.0f;
        weight[i] = 0.0f;
    }
    if (i < nt) counts[i] = 0u;
}

// First tile of a work-group's window of min(nt, kSplatLdsTiles): around the
// tile of a particle in its middle.
template <int ALG>
__device__ __forceinline__ uint32_t splat_window(const PGrid& g, uint32_t np, const float* __restrict__ pos, uint32_t base,
                                                 uint32_t nt) {
    if (nt <= kSplatLdsTiles) return 0;
    const uint32_t p = base + kBlock * kSplatItems / 2;
    const uint32_t t = splat_at<ALG>(g, pos, p < np ? p : np - 1).tile;
    return t < kSplatLdsTiles / 2 ? 0 : min(t - kSplatLdsTiles / 2, nt - kSplatLdsTiles);
}

// The lanes of the wave with `on` and this lane's tile (0 where not on).
__device__ __forceinline__ uint64_t same_tile(bool on, uint32_t tile) {
    uint64_t mine = 0;
    for (uint64_t todo = __ballot(on); todo;) {
        const uint32_t t = uint32_t(__builtin_amdgcn_readlane(int(tile), __ffsll((unsigned long long)todo) - 1));
        const uint64_t same = __ballot(on && tile == t);
        if (on && tile == t) mine = same;
        todo &= ~same;
    }
    return mine;
}
__device__ __forceinline__ uint32_t rank_in(uint64_t lanes) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(lanes >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(lanes), 0u));
}

// counts[t] += this work-group's particles of tile t.  Dynamic LDS: the window.
template <int ALG>
__global__ void __launch_bounds__(kBlock) k_splat_count(PGrid g, uint32_t np, const float* __restrict__ pos,
                                                        uint32_t* counts, uint32_t nt) {
    extern __shared__ uint32_t hist[];
    const uint32_t base = blockIdx.x * (kBlock * kSplatItems);
    const uint32_t win = min(nt, kSplatLdsTiles), lo = splat_window<ALG>(g, np, pos, base, nt);
    for (uint32_t i = threadIdx.x; i < win; i += kBlock) hist[i] = 0u;
    __syncthreads();
    if (win == nt) {
#pragma unroll 4
        for (uint32_t j = 0; j < kSplatItems; ++j) {
            const uint32_t p = base + j * kBlock + threadIdx.x;
            if (p < np) atomicAdd(&hist[splat_at<ALG>(g, pos, p).tile], 1u);
        }
    } else {
        for (uint32_t j = 0; j < kSplatItems; ++j) {
            if (base + j * kBlock >= np) break;   // the same for every work-item
            const uint32_t p = base + j * kBlock + threadIdx.x;
            const uint32_t t = splat_at<ALG>(g, pos, p < np ? p : np - 1).tile;
            if (p < np && t - lo < win) atomicAdd(&hist[t - lo], 1u);
            const uint64_t mine = same_tile(p < np && t - lo >= win, t);
            if (mine && rank_in(mine) == 0) atomicAdd(&counts[t], uint32_t(__popcll(mine)));
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < win; i += kBlock)
        if (hist[i]) atomicAdd(&counts[lo + i], hist[i]);
}

// One work-group: counts -> start (exclusive prefix, start[nt] = the total)
// and cursor, and the chunks in tile order: work[2 j] = tile, work[2 j + 1] =
// its first sorted particle; *nwork = their number.  counts is 16-byte aligned
// and readable up to the next multiple of four words.
__global__ void __launch_bounds__(1024) k_splat_scan(uint32_t nt, const uint32_t* __restrict__ counts,
                                                     uint32_t* __restrict__ start, uint32_t* __restrict__ cursor,
                                                     uint32_t* __restrict__ work, uint32_t* __restrict__ nwork) {
    __shared__ uint32_t sp[16], sc[16];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint32_t run = 0, w = 0;   // particles and chunks of the tiles before
    for (uint32_t b = 0; b < nt; b += 4096) {
        const uint32_t i = b + 4 * t;
        uint4 c4 = make_uint4(0u, 0u, 0u, 0u);
        if (i < nt) c4 = *reinterpret_cast<const uint4*>(counts + i);
        const uint32_t c[4] = {c4.x, i + 1 < nt ? c4.y : 0u, i + 2 < nt ? c4.z : 0u, i + 3 < nt ? c4.w : 0u};
        uint32_t ip = 0, ic = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            ip += c[k];
            ic += (c[k] + kSplatChunk - 1) / kSplatChunk;
        }
        const uint32_t mp = ip, mc = ic;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t up = uint32_t(__shfl_up(int(ip), o, 64)), uc = uint32_t(__shfl_up(int(ic), o, 64));
            if (lane >= uint32_t(o)) {
                ip += up;
                ic += uc;
            }
        }
        if (lane == 63) {
            sp[wave] = ip;
            sc[wave] = ic;
        }
        __syncthreads();
        uint32_t q = run + ip - mp, j = w + ic - mc;
#pragma unroll
        for (uint32_t v = 0; v < 16; ++v) {
            const uint32_t vp = sp[v], vc = sc[v];
            if (v < wave) {
                q += vp;
                j += vc;
            }
            run += vp;
            w += vc;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            if (i + k >= nt) break;
            start[i + k] = q;
            cursor[i + k] = q;
            for (uint32_t e = 0; e < c[k]; e += kSplatChunk, ++j) {
                work[2 * size_t(j)] = i + k;
                work[2 * size_t(j) + 1] = q + e;
            }
            q += c[k];
        }
    }
    if (t == 0) {
        start[nt] = run;
        *nwork = w;
    }
}

// order = the particles by tile.  A work-group ranks its particles of a tile
// in LDS and reserves their slots with one atomic a tile (outside the window a
// wave does).
template <int ALG>
__global__ void __launch_bounds__(kBlock) k_splat_order(PGrid g, uint32_t np, const float* __restrict__ pos,
                                                        uint32_t* cursor, uint32_t* __restrict__ order, uint32_t nt) {
    extern __shared__ uint32_t hist[];
    const uint32_t base = blockIdx.x * (kBlock * kSplatItems);
    const uint32_t win = min(nt, kSplatLdsTiles), lo = splat_window<ALG>(g, np, pos, base, nt);
    for (uint32_t i = threadIdx.x; i < win; i += kBlock) hist[i] = 0u;
    __syncthreads();
    uint32_t tile[kSplatItems], rank[kSplatItems];   // tile: in the window
#pragma unroll
    for (uint32_t j = 0; j < kSplatItems; ++j) {
        tile[j] = ~0u;
        if (base + j * kBlock >= np) continue;   // the same for every work-item
        const uint32_t p = base + j * kBlock + threadIdx.x;
        const uint32_t t = splat_at<ALG>(g, pos, p < np ? p : np - 1).tile;
        if (p < np) tile[j] = t - lo;
        rank[j] = tile[j] < win ? atomicAdd(&hist[tile[j]], 1u) : 0u;
        if (win < nt) {
            const uint64_t mine = same_tile(p < np && tile[j] >= win, t);
            const uint32_t r = rank_in(mine);
            uint32_t at = 0;
            if (mine && r == 0) at = atomicAdd(&cursor[t], uint32_t(__popcll(mine)));
            at = uint32_t(__shfl(int(at), mine ? __ffsll((unsigned long long)mine) - 1 : 0, 64));
            if (mine) order[at + r] = p;
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < win; i += kBlock)
        if (hist[i]) hist[i] = atomicAdd(&cursor[lo + i], hist[i]);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kSplatItems; ++j) {
        const uint32_t p = base + j * kBlock + threadIdx.x;
        if (tile[j] < win) order[hist[tile[j]] + rank[j]] = p;
    }
}

template <int ALG>
__global__ void __launch_bounds__(kSplatBlock) k_splat_tiles(PGrid g, const float* __restrict__ pos,
                                                             const float* __restrict__ val, int span, int off,
                                                             const uint32_t* __restrict__ start,
                                                             const uint32_t* __restrict__ order,
                                                             const uint32_t* __restrict__ work,
                                                             const uint32_t* __restrict__ nwork,
                                                             float* __restrict__ field, float* __restrict__ weight) {
    constexpr int N = splat_corners(ALG), E = kTileEdge + N - 1, kWaves = kSplatBlock / 64;
    __shared__ float4 part[kSplatChunk];                 // position and value, by cell
    __shared__ uint32_t first[kSplatBlock], wsum[kWaves];
    __shared__ float sv[E * E * E], sw[E * E * E];
    if (blockIdx.x >= *nwork) return;
    const int t = threadIdx.x;
    for (int i = t; i < E * E * E; i += kSplatBlock) sv[i] = sw[i] = 0.0f;
    first[t] = 0u;
    const uint32_t tile = work[2 * size_t(blockIdx.x)], q0 = work[2 * size_t(blockIdx.x) + 1];
    const uint32_t n = min(start[tile + 1] - q0, kSplatChunk);
    __syncthreads();
    float4 v[kSplatRounds];
    uint32_t cell[kSplatRounds], rank[kSplatRounds];
#pragma unroll
    for (uint32_t j = 0; j < kSplatRounds; ++j) {
        const uint32_t q = j * kSplatBlock + t;
        cell[j] = rank[j] = 0u;
        if (q < n) {
            const size_t p = order[q0 + q];
            v[j] = make_float4(pos[3 * p], pos[3 * p + 1], pos[3 * p + 2], val[size_t(span) * p + size_t(off)]);
            cell[j] = splat_at<ALG>(g, v[j].x, v[j].y, v[j].z).cell;
            rank[j] = atomicAdd(&first[cell[j]], 1u);
        }
    }
    __syncthreads();
    // counts -> exclusive prefix
    const uint32_t mine = first[t];
    uint32_t incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = uint32_t(__shfl_up(int(incl), o, 64));
        if ((t & 63) >= o) incl += u;
    }
    // with bit 31: a cell of the wave holds more than kSplatCell
    const bool crowded = __any(mine > kSplatCell);
    if ((t & 63) == 63) wsum[t >> 6] = incl | (crowded ? 1u << 31 : 0u);
    __syncthreads();
    uint32_t q = incl - mine, dense = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t u = wsum[w];
        q += w < (t >> 6) ? u & 0x7fffffffu : 0u;
        dense |= u >> 31;
    }
    first[t] = q;   // as it stays
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kSplatRounds; ++j)
        if (j * kSplatBlock + t < n) part[first[cell[j]] + rank[j]] = v[j];
    __syncthreads();
    // this work-item's cell: its particles' sums per corner
    float av[N * N * N], aw[N * N * N];
#pragma unroll
    for (int k = 0; k < N * N * N; ++k) av[k] = aw[k] = 0.0f;
    auto add = [&](const float4& s) {
        if constexpr (ALG == MGF_PG_P2GSUM) {
            av[0] += s.w;
        } else {
            PStencil st;
            pg_stencil(g, s.x, s.y, s.z, ALG, st);
            float w[3][N];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const bool skip = ALG == MGF_PG_QUADRATIC && st.w[a][0] == 0.0f;
#pragma unroll
                for (int k = 0; k < N; ++k) w[a][k] = skip ? st.w[a][k + (N < 4 ? 1 : 0)] : st.w[a][k];
            }
            // a value that is not finite makes NaN of the +0 weights left
            // out: all of its 64 corners go straight to the field
            if (ALG == MGF_PG_QUADRATIC && !(fabsf(s.w) <= MGF_UNKNOWN)) {
                for_corners<4>(g, st, [&](uint32_t node, float wt) {
                    atomicAdd(&field[node], wt * s.w);
                    atomicAdd(&weight[node], wt);
                });
                return;
            }
#pragma unroll
            for (int z = 0; z < N; ++z)
#pragma unroll
                for (int y = 0; y < N; ++y)
#pragma unroll
                    for (int x = 0; x < N; ++x) {
                        const float wt = w[0][x] * w[1][y] * w[2][z];
                        av[(z * N + y) * N + x] += wt * s.w;
                        aw[(z * N + y) * N + x] += wt;
                    }
        }
    };
    // LDS place of corner k of the cell with lowest node `at`
    auto corner = [](int at, int k) { return at + ((k / (N * N)) * E + (k / N) % N) * E + k % N; };
    auto node_of = [](uint32_t c) {
        return ((int(c) / (kTileEdge * kTileEdge)) * E + (int(c) / kTileEdge) % kTileEdge) * E + int(c) % kTileEdge;
    };
    for (const uint32_t q1 = q + min(mine, kSplatCell); q < q1; ++q) add(part[q]);
    const int at = node_of(uint32_t(t));
#pragma unroll
    for (int k = 0; k < N * N * N; ++k) {
        if (mine) {
            sv[corner(at, k)] += av[k];
            if (ALG != MGF_PG_P2GSUM) sw[corner(at, k)] += aw[k];
        }
        __syncthreads();
    }
    // Cells of more than kSplatCell particles: a work-item sums the rest of
    // kSplatRounds consecutive ones and adds them to the tile by atomics, once
    // a cell.
    if (dense) {
        uint32_t cur = ~0u;
        auto flush = [&]() {
            if (cur == ~0u) return;
            const int o = node_of(cur);
#pragma unroll
            for (int k = 0; k < N * N * N; ++k) {
                atomicAdd(&sv[corner(o, k)], av[k]);
                if (ALG != MGF_PG_P2GSUM) atomicAdd(&sw[corner(o, k)], aw[k]);
            }
        };
        const uint32_t b = uint32_t(t) * kSplatRounds, e = min(n, b + kSplatRounds);
        for (uint32_t i = b; i < e; ++i) {
            const float4 s = part[i];
            const uint32_t c = splat_at<ALG>(g, s.x, s.y, s.z).cell;
            if (i - first[c] < kSplatCell) continue;
            if (c != cur) {
                flush();
                cur = c;
#pragma unroll
                for (int k = 0; k < N * N * N; ++k) av[k] = aw[k] = 0.0f;
            }
            add(s);
        }
        flush();
        __syncthreads();
    }
    const uint32_t ntx = splat_tiles(g.nx, N), nty = splat_tiles(g.ny, N);
    const int bx = int(tile % ntx) * kTileEdge - (N - 1), by = int((tile / ntx) % nty) * kTileEdge - (N - 1),
              bz = int(tile / (ntx * nty)) * kTileEdge - (N - 1);
    for (int i = t; i < E * E * E; i += kSplatBlock) {
        const float a = sv[i], w = sw[i];
        if (a == 0.0f && w == 0.0f) continue;
        const uint32_t node = pg_index(g, bx + i % E, by + (i / E) % E, bz + i / (E * E));
        atomicAdd(&field[node], a);
        if (ALG != MGF_PG_P2GSUM) atomicAdd(&weight[node], w);
    }
}

// The same sums without a sort: a work-group's particles are merged in an LDS
// hash table by node (those of a set in cell order are neighbours and share
// the nodes of their supports), and the flush issues one global atomic a
// distinct node.  A contribution that finds no slot within kProbe probes goes
// straight to global memory.
constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;
constexpr int kProbe = 32;

template <int HB>
__device__ __forceinline__ void lds_accumulate(uint32_t* keys, float* sv, float* sw, uint32_t key, float a, float b,
                                               bool with_w, float* gf, float* gw) {
    constexpr uint32_t T = 1u << HB;
    uint32_t h = (key * 2654435761u) >> (32 - HB);
    for (int probe = 0; probe < kProbe; ++probe) {
        // a slot once claimed keeps its key: read first, claim empty slots only
        uint32_t k = __atomic_load_n(&keys[h], __ATOMIC_RELAXED);
        if (k == kEmptyKey) k = atomicCAS(&keys[h], kEmptyKey, key);
        if (k == kEmptyKey || k == key) {
            atomicAdd(&sv[h], a);
            if (with_w) atomicAdd(&sw[h], b);
            return;
        }
        h = (h + 1) & (T - 1);
    }
    atomicAdd(gf, a);
    if (with_w) atomicAdd(gw, b);
}

// Tables of 1024 slots for P2GSUM and LINEAR (8 nodes a particle), 2048 for
// the 64-node supports.
template <int ALG>
__global__ void __launch_bounds__(kBlock) k_p2g_hash(PGrid g, int64_t np, const float* __restrict__ pos,
                                                     const float* __restrict__ val, int span, int off,
                                                     float* __restrict__ field, float* __restrict__ weight) {
    constexpr int HB = ALG == MGF_PG_P2GSUM || ALG == MGF_PG_LINEAR ? 10 : 11;
    constexpr uint32_t T = 1u << HB;
    __shared__ uint32_t keys[T];
    __shared__ float sv[T], sw[T];
    for (uint32_t i = threadIdx.x; i < T; i += kBlock) {
        keys[i] = kEmptyKey;
        sv[i] = 0.0f;
        sw[i] = 0.0f;
    }
    __syncthreads();
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p < np) {
        const float px = pos[3 * p], py = pos[3 * p + 1], pz = pos[3 * p + 2], v = val[int64_t(span) * p + off];
        if constexpr (ALG == MGF_PG_P2GSUM) {
            const uint32_t node = pos_cell(g, px, py, pz);
            lds_accumulate<HB>(keys, sv, sw, node, v, 0.0f, false, &field[node], nullptr);
        } else {
            PStencil st;
            pg_stencil(g, px, py, pz, ALG, st);
            constexpr int N = ALG == MGF_PG_LINEAR ? 2 : 4, lo = N == 2 ? 0 : -1;
#pragma unroll 1
            for (int k = 0; k < N * N * N; ++k) {
                const int x = k % N, y = (k / N) % N, z = k / (N * N);
                const uint32_t node = pg_index(g, st.i0[0] + x + lo, st.i0[1] + y + lo, st.i0[2] + z + lo);
                const float wt = st.w[0][x] * st.w[1][y] * st.w[2][z];
                lds_accumulate<HB>(keys, sv, sw, node, wt * v, wt, true, &field[node], &weight[node]);
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < T; i += kBlock) {
        const uint32_t k = keys[i];
        if (k == kEmptyKey) continue;
        atomicAdd(&field[k], sv[i]);
        if (ALG != MGF_PG_P2GSUM) atomicAdd(&weight[k], sw[i]);
    }
}

// normalizeCCSField (EulerParticlesTool.cu:290-308).
__global__ void __launch_bounds__(kBlock) k_p2g_normalize(size_t n, float* __restrict__ field,
                                                          const float* __restrict__ weight) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n && weight[i] > 0.0f) field[i] /= weight[i];
}

// The value of one field at a particle: summed from 0 in corner order
// z, y, x (G2PNEAREST: the value of its cell).  A row of N corners that lies
// inside the grid is one wide load (4-byte aligned): particles in loose order
// make every lane's load a cache line of its own, so the loads, not the sums,
// bound the kernel (QUADRATIC, 1.23M particles: 115 us with one load a
// corner, 56 us this way; k_transfer_vel<2> of 5.0M: 207 -> 154 us).  Rows that cross the grid's ends clamp corner
// by corner.
template <int N>
__device__ __forceinline__ float g2p_one(const PGrid& g, float px, float py, float pz, const float* __restrict__ f,
                                         int alg) {
    if (alg == MGF_PG_G2PNEAREST) return f[pos_cell(g, px, py, pz)];
    constexpr int lo = N == 2 ? 0 : -1;
    PStencil st;
    pg_stencil(g, px, py, pz, alg, st);
    typedef float Row __attribute__((ext_vector_type(N)));
    typedef float RowAt __attribute__((ext_vector_type(N), aligned(4)));
    Row r[N][N];
    const int x0 = st.i0[0] + lo;
    const bool inside = x0 >= 0 && x0 <= g.nx - N;
#pragma unroll
    for (int z = 0; z < N; ++z)
#pragma unroll
        for (int y = 0; y < N; ++y) {
            if (inside) {
                r[z][y] = *reinterpret_cast<const RowAt*>(f + pg_index(g, x0, st.i0[1] + y + lo, st.i0[2] + z + lo));
            } else {
#pragma unroll
                for (int x = 0; x < N; ++x) r[z][y][x] = f[pg_index(g, x0 + x, st.i0[1] + y + lo, st.i0[2] + z + lo)];
            }
        }
    float acc = 0.0f;
#pragma unroll
    for (int z = 0; z < N; ++z)
#pragma unroll
        for (int y = 0; y < N; ++y)
#pragma unroll
            for (int x = 0; x < N; ++x) acc += st.w[0][x] * st.w[1][y] * st.w[2][z] * r[z][y][x];
    return acc;
}

// accumulateCCSField2Particles (EulerParticlesTool.cu:198-288): summed from
// 0 in corner order z, y, x.
template <int N>
__global__ void __launch_bounds__(kBlock) k_g2p(PGrid g, int64_t np, const float* __restrict__ pos,
                                                const float* __restrict__ field, int alg, float* val, int span,
                                                int off) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    const float px = pos[3 * p], py = pos[3 * p + 1], pz = pos[3 * p + 2];
    val[int64_t(span) * p + off] =
        (alg == MGF_PG_G2PNEAREST || alg == MGF_PG_LINEAR || alg == MGF_PG_QUADRATIC || alg == MGF_PG_CUBIC)
            ? g2p_one<N>(g, px, py, pz, field, alg) : 0.0f;
}


// The particle-velocity update of the three solvers in one pass, with the
// operations and rounding of the reference's separate calls:
//   PIC  (ParticleInCell.cpp:101):  v = G2P(in)
//   FLIP (FluidImplicitParticle.cpp:109-110): v = fma(1, G2P(delta), v)
//   MIX  (MixPICAndFLIP.cpp:114-129): p = G2P(in); v = fma(1, G2P(delta), v);
//        v = keep * v; v = fma(mixing, p, v)
struct Faces3 {
    const float* f[3];
};
template <int N>
__device__ __forceinline__ void transfer_one(const PGrid& g, float px, float py, float pz, const float* fin,
                                             const float* fdelta, int kind, int alg, float keep, float mixing,
                                             float* v) {
    if (kind == MGF_PSOLVER_PIC) {
        *v = g2p_one<N>(g, px, py, pz, fin, alg);
        return;
    }
    const float pic = kind == MGF_PSOLVER_MIX ? g2p_one<N>(g, px, py, pz, fin, alg) : 0.0f;
    float u = __builtin_fmaf(1.0f, g2p_one<N>(g, px, py, pz, fdelta, alg), *v);
    if (kind == MGF_PSOLVER_MIX) u = __builtin_fmaf(mixing, pic, keep * u);
    *v = u;
}

template <int N>
__global__ void __launch_bounds__(kBlock) k_transfer_vel(PGrid g0, PGrid g1, PGrid g2, int64_t np,
                                                         const float* __restrict__ pos, Faces3 in, Faces3 delta,
                                                         int kind, int alg, float keep, float mixing,
                                                         float* __restrict__ vel) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    const float px = pos[3 * p], py = pos[3 * p + 1], pz = pos[3 * p + 2];
    transfer_one<N>(g0, px, py, pz, in.f[0], delta.f[0], kind, alg, keep, mixing, &vel[3 * p]);
    transfer_one<N>(g1, px, py, pz, in.f[1], delta.f[1], kind, alg, keep, mixing, &vel[3 * p + 1]);
    transfer_one<N>(g2, px, py, pz, in.f[2], delta.f[2], kind, alg, keep, mixing, &vel[3 * p + 2]);
}

// max over the work-group, then one atomic per work-group.
__device__ __forceinline__ void block_max_atomic(uint32_t m, uint32_t* out) {
    __shared__ uint32_t wmax[kBlock / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), o, 64)));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t b = wmax[0];
#pragma unroll
        for (int q = 1; q < kBlock / 64; ++q) b = max(b, wmax[q]);
        atomicMax(out, b);
    }
}

// One particle advection substep in one pass (EulerParticles.cpp:273-313:
// the axpys of RK1/2/3 with the samples between them, same order and
// rounding), v1 = the velocity sampled at the positions it starts from.  With
// resample, the velocity at the new positions is written to v1 and its
// largest magnitude to vmax_bits, for the next substep's length.
__global__ void __launch_bounds__(kBlock) k_rk_substep(GridDev g, Vel V, int64_t np, float* __restrict__ pos,
                                                       float* __restrict__ v1, int order, float step, float half,
                                                       float three_q, float c1, float c2, float c3, int resample,
                                                       uint32_t* vmax_bits) {
    uint32_t m = 0;
    const int64_t stride = int64_t(gridDim.x) * kBlock;
    for (int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x; p < np; p += stride) {
        const float x0 = pos[3 * p], y0 = pos[3 * p + 1], z0 = pos[3 * p + 2];
        const float ax = v1[3 * p], ay = v1[3 * p + 1], az = v1[3 * p + 2];
        float x, y, z;
        if (order == 1) {
            x = __builtin_fmaf(step, ax, x0); y = __builtin_fmaf(step, ay, y0); z = __builtin_fmaf(step, az, z0);
        } else if (order == 2) {
            float bx, by, bz;
            sample_vel_any(V, g, __builtin_fmaf(half, ax, x0), __builtin_fmaf(half, ay, y0), __builtin_fmaf(half, az, z0),
                       bx, by, bz);
            x = __builtin_fmaf(step, bx, x0); y = __builtin_fmaf(step, by, y0); z = __builtin_fmaf(step, bz, z0);
        } else if (order == 3) {
            float bx, by, bz, cx, cy, cz;
            sample_vel_any(V, g, __builtin_fmaf(half, ax, x0), __builtin_fmaf(half, ay, y0), __builtin_fmaf(half, az, z0),
                       bx, by, bz);
            sample_vel_any(V, g, __builtin_fmaf(three_q, bx, x0), __builtin_fmaf(three_q, by, y0),
                       __builtin_fmaf(three_q, bz, z0), cx, cy, cz);
            x = __builtin_fmaf(c3, cx, __builtin_fmaf(c2, bx, __builtin_fmaf(c1, ax, x0)));
            y = __builtin_fmaf(c3, cy, __builtin_fmaf(c2, by, __builtin_fmaf(c1, ay, y0)));
            z = __builtin_fmaf(c3, cz, __builtin_fmaf(c2, bz, __builtin_fmaf(c1, az, z0)));
        } else {
            x = x0; y = y0; z = z0;
        }
        pos[3 * p] = x; pos[3 * p + 1] = y; pos[3 * p + 2] = z;
        if (resample) {
            float a, b, c;
            sample_vel_any(V, g, x, y, z, a, b, c);
            v1[3 * p] = a; v1[3 * p + 1] = b; v1[3 * p + 2] = c;
            m = max(m, max(__float_as_uint(fabsf(a)), max(__float_as_uint(fabsf(b)), __float_as_uint(fabsf(c)))));
        }
    }
    if (resample) block_max_atomic(m, vmax_bits);
}

// The velocity at each particle and its largest magnitude (the first
// sample of a substep loop).
__global__ void __launch_bounds__(kBlock) k_sample_absmax(GridDev g, Vel V, int64_t np, const float* __restrict__ pos,
                                                          float* __restrict__ out, uint32_t* vmax_bits) {
    uint32_t m = 0;
    const int64_t stride = int64_t(gridDim.x) * kBlock;
    for (int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x; p < np; p += stride) {
        float a, b, c;
        sample_vel_any(V, g, pos[3 * p], pos[3 * p + 1], pos[3 * p + 2], a, b, c);
        out[3 * p] = a; out[3 * p + 1] = b; out[3 * p + 2] = c;
        m = max(m, max(__float_as_uint(fabsf(a)), max(__float_as_uint(fabsf(b)), __float_as_uint(fabsf(c)))));
    }
    block_max_atomic(m, vmax_bits);
}

// statisticalFluidDensity (EulerParticlesTool.cu:27-46): +1 per particle.
__global__ void __launch_bounds__(kBlock) k_particle_counts(PGrid g, int64_t np, const float* __restrict__ pos,
                                                            float* out) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    atomicAdd(&out[pos_cell(g, pos[3 * p], pos[3 * p + 1], pos[3 * p + 2])], 1.0f);
}

// buildFluidMarkers (EulerParticlesTool.cu:48-77): 2 solid, 1 with a
// particle, 0 else.
__global__ void __launch_bounds__(kBlock) k_particle_markers(size_t n, const float* __restrict__ solid,
                                                             float* __restrict__ io) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i >= n) return;
    io[i] = solid[i] < 0.0f ? 2.0f : (io[i] > 0.0f ? 1.0f : 0.0f);
}

// axpyReal (ThrustWapper.cu:281-292, cuBLAS axpy): y = a x + y as one fused
// multiply-add; scaleReal (:294-304): x = a x.
__global__ void __launch_bounds__(kBlock) k_axpy_n(size_t n, float a, const float* __restrict__ x, float* y) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n) y[i] = __builtin_fmaf(a, x[i], y[i]);
}
__global__ void __launch_bounds__(kBlock) k_scale_n(size_t n, float a, float* x) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n) x[i] = a * x[i];
}

// fixParticlesPosWithBoundarys (EulerParticlesTool.cu:310-333, 870-894):
// positions clamped to the grid box; the reference launches one work-item per
// cell, so only the first min(cells, particles) particles are clamped.
__global__ void __launch_bounds__(kBlock) k_clamp_particles(int64_t m, float* pos, float lx, float ly, float lz,
                                                            float hx, float hy, float hz) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= m) return;
    pos[3 * p] = fmaxf(lx, fminf(pos[3 * p], hx));
    pos[3 * p + 1] = fmaxf(ly, fminf(pos[3 * p + 1], hy));
    pos[3 * p + 2] = fmaxf(lz, fminf(pos[3 * p + 2], hz));
}

// ---- particle generation (generateParticlesInFluid, EulerParticles.cpp:
// 163-201; findFluidGrid, EulerParticlesTool.cu:5-25) -----------------------
// A tile of kGenTile consecutive cells per work-group: the count pass sums the
// fluid cells of each tile, one work-group scans the tile sums, and the emit
// pass ranks the fluid cells inside its tile (wave ballots, x-fastest order)
// and writes their particles.
constexpr int kGenRows = 8;
constexpr int kGenTile = kBlock * kGenRows;

__device__ __forceinline__ bool fluid_cell(const float* fluid, const float* solid, size_t c) {
    return fluid[c] < 0.0f && !(solid && solid[c] < 0.0f);
}

// Fluid cells of this work-group's tile among rows [0, kGenRows): for each row
// the rank of this work-item's cell among the row's fluid cells and the row
// total.  wsum holds one count per wave.
__device__ __forceinline__ void row_rank(bool f, uint32_t* wsum, uint32_t& before, uint32_t& total) {
    const uint64_t b = __ballot(f);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wsum[wave] = uint32_t(__popcll(b));
    __syncthreads();
    uint32_t pre = uint32_t(__popcll(b & ((uint64_t(1) << lane) - 1)));
    total = 0;
#pragma unroll
    for (int q = 0; q < kBlock / 64; ++q) {
        if (q < wave) pre += wsum[q];
        total += wsum[q];
    }
    before = pre;
    __syncthreads();
}

__global__ void __launch_bounds__(kBlock) k_gen_count(size_t n, const float* __restrict__ fluid,
                                                      const float* __restrict__ solid, uint32_t* __restrict__ tiles) {
    __shared__ uint32_t wsum[kBlock / 64];
    const size_t base = size_t(blockIdx.x) * kGenTile;
    uint32_t sum = 0;
    for (int j = 0; j < kGenRows; ++j) {
        const size_t c = base + size_t(j) * kBlock + threadIdx.x;
        uint32_t before, total;
        row_rank(c < n && fluid_cell(fluid, solid, c), wsum, before, total);
        sum += total;
    }
    if (threadIdx.x == 0) tiles[blockIdx.x] = sum;
}

// In place: tiles[0..nt) -> exclusive prefix sums, tiles[nt] = the total.
__global__ void __launch_bounds__(1024) k_gen_scan(uint32_t nt, uint32_t* tiles) {
    __shared__ uint32_t part[1024];
    const uint32_t t = threadIdx.x, per = (nt + 1023) / 1024;
    const uint32_t b = min(nt, t * per), e = min(nt, b + per);
    uint32_t s = 0;
    for (uint32_t i = b; i < e; ++i) s += tiles[i];
    part[t] = s;
    __syncthreads();
    for (uint32_t o = 1; o < 1024; o <<= 1) {   // inclusive Hillis-Steele scan
        const uint32_t v = t >= o ? part[t - o] : 0u;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    uint32_t run = t ? part[t - 1] : 0u;
    for (uint32_t i = b; i < e; ++i) {
        const uint32_t v = tiles[i];
        tiles[i] = run;
        run += v;
    }
    if (t == 1023) tiles[nt] = part[1023];
}

// SplitMix64's output function (Steele, Lea, Flood, "Fast splittable
// pseudorandom number generators", OOPSLA 2014).
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float particle_jitter(uint64_t seed, uint64_t index, int axis) {
    return float(splitmix64(seed ^ splitmix64(3 * index + uint64_t(axis))) >> 40) * (1.0f / 16777216.0f);
}

__global__ void __launch_bounds__(kBlock) k_gen_emit(GridDev g, size_t n, const float* __restrict__ fluid,
                                                     const float* __restrict__ solid,
                                                     const uint32_t* __restrict__ tiles, int per_cell, uint64_t seed,
                                                     float* __restrict__ pos) {
    __shared__ uint32_t wsum[kBlock / 64];
    const size_t base = size_t(blockIdx.x) * kGenTile;
    uint32_t rank = tiles[blockIdx.x];
    for (int j = 0; j < kGenRows; ++j) {
        const size_t c = base + size_t(j) * kBlock + threadIdx.x;
        const bool f = c < n && fluid_cell(fluid, solid, c);
        uint32_t before, total;
        row_rank(f, wsum, before, total);
        if (f) {
            const uint32_t x = uint32_t(c % uint32_t(g.nx));
            const uint32_t y = uint32_t((c / uint32_t(g.nx)) % uint32_t(g.ny));
            const uint32_t z = uint32_t(c / (size_t(g.nx) * uint32_t(g.ny)));
            const uint64_t first = uint64_t(rank + before) * uint64_t(per_cell);
            for (int i = 0; i < per_cell; ++i) {
                const uint64_t idx = first + uint64_t(i);
                pos[3 * idx] = (float(x) + particle_jitter(seed, idx, 0)) * g.hx + g.ox;
                pos[3 * idx + 1] = (float(y) + particle_jitter(seed, idx, 1)) * g.hy + g.oy;
                pos[3 * idx + 2] = (float(z) + particle_jitter(seed, idx, 2)) * g.hz + g.oz;
            }
        }
        rank += total;
    }
}

// m_DeltaGridVelField.plusAlphaX(in, -1); m_DeltaGridVelField *= -1
// (FluidImplicitParticle.cpp:105-106): one axpy with alpha -1, then a sign flip.
__global__ void __launch_bounds__(kBlock) k_flip_delta(size_t n, const float* __restrict__ in, float* delta) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n) delta[i] = -__builtin_fmaf(-1.0f, in[i], delta[i]);
}

// Pressure markers from particles (buildFluidMarkers, EulerParticlesTool.cu:
// 48-77): 2 in solid cells, then 1 in every other cell holding a particle.
__global__ void __launch_bounds__(kBlock) k_markers_solid(size_t n, const uint8_t* __restrict__ solid_mask,
                                                          uint8_t* __restrict__ markers) {
    const size_t i = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (i < n) markers[i] = solid_mask[i] ? uint8_t(2) : uint8_t(0);
}
__global__ void __launch_bounds__(kBlock) k_markers_particles(PGrid g, int64_t np, const float* __restrict__ pos,
                                                              uint8_t* markers) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    const uint32_t c = pos_cell(g, pos[3 * p], pos[3 * p + 1], pos[3 * p + 2]);
    if (markers[c] != 2) markers[c] = 1;
}

// ---- the particle-to-grid splat as a gather over binned particles ---------
// Particles are counting-sorted by the lower corner s of their support on the
// cell grid (s = floor((p - o)/h - 1/2) per axis, clamped to [-1, n-1]: bins
// (nx+1)(ny+1)(nz+1)).  A node of a target grid (the cells, or the faces of
// one axis) then sums, with no atomics, over the particles of the bins whose
// supports can reach it: on the target grid a node i receives from supports
// with lower corner in [i - lo - n + 1, i - lo] (lo, n: the kernel's corner
// offset and width), and on the axis the target grid is shifted along, that
// corner is the cell grid's or the next one (the same floor taken half a cell
// further), so one more bin is visited there.  Each visited particle's
// support on the target grid is evaluated as in the per-particle splat; the
// corners that clamp onto the node add their weights.
struct BinGrid {
    int nx, ny, nz;   // cells of the grid the bins follow
};

__device__ __forceinline__ uint32_t bin_of(const PGrid& c, float px, float py, float pz) {
    const float rel[3] = {px - c.ox - c.hx * 0.5f, py - c.oy - c.hy * 0.5f, pz - c.oz - c.hz * 0.5f};
    const float h[3] = {c.hx, c.hy, c.hz};
    const float rh[3] = {c.rhx, c.rhy, c.rhz};
    const int n[3] = {c.nx, c.ny, c.nz};
    uint32_t b[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int s = floor_ref(div_h(rel[k], h[k], rh[k], c.pow2));
        s = s < -1 ? -1 : (s > n[k] - 1 ? n[k] - 1 : s);
        b[k] = uint32_t(s + 1);
    }
    return (b[2] * uint32_t(c.ny + 1) + b[1]) * uint32_t(c.nx + 1) + b[0];
}

__global__ void __launch_bounds__(kBlock) k_bin_count(PGrid c, int64_t np, const float* __restrict__ pos,
                                                      uint32_t* counts) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    atomicAdd(&counts[bin_of(c, pos[3 * p], pos[3 * p + 1], pos[3 * p + 2])], 1u);
}

// Tile sums of a u32 array (kGenTile entries per work-group).
__global__ void __launch_bounds__(kBlock) k_scan_tiles(size_t n, const uint32_t* __restrict__ a,
                                                       uint32_t* __restrict__ tiles) {
    __shared__ uint32_t wsum[kBlock / 64];
    const size_t base = size_t(blockIdx.x) * kGenTile + size_t(threadIdx.x) * kGenRows;
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kGenRows; ++j)
        if (base + j < n) sum += a[base + j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += uint32_t(__shfl_xor(int(sum), o, 64));
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
#pragma unroll
        for (int q = 0; q < kBlock / 64; ++q) t += wsum[q];
        tiles[blockIdx.x] = t;
    }
}

// start[i] = exclusive prefix of a (tile offsets already scanned), and a copy
// in cursor; start[n] = the total.
__global__ void __launch_bounds__(kBlock) k_scan_apply(size_t n, const uint32_t* __restrict__ a,
                                                       const uint32_t* __restrict__ tiles, uint32_t nt,
                                                       uint32_t* __restrict__ start, uint32_t* __restrict__ cursor) {
    __shared__ uint32_t part[kBlock];
    const size_t base = size_t(blockIdx.x) * kGenTile + size_t(threadIdx.x) * kGenRows;
    uint32_t v[kGenRows], sum = 0;
#pragma unroll
    for (int j = 0; j < kGenRows; ++j) {
        v[j] = base + j < n ? a[base + j] : 0u;
        sum += v[j];
    }
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < kBlock; o <<= 1) {   // inclusive scan of the work-items' sums
        const uint32_t t = threadIdx.x >= uint32_t(o) ? part[threadIdx.x - o] : 0u;
        __syncthreads();
        part[threadIdx.x] += t;
        __syncthreads();
    }
    uint32_t run = tiles[blockIdx.x] + (threadIdx.x ? part[threadIdx.x - 1] : 0u);
#pragma unroll
    for (int j = 0; j < kGenRows; ++j) {
        if (base + j < n) {
            start[base + j] = run;
            cursor[base + j] = run;
        }
        run += v[j];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) start[n] = tiles[nt];
}

// Each particle's slot in bin order, with sorted copies of its position and
// (when vel is given) its velocity, so the splat reads them contiguously.
__global__ void __launch_bounds__(kBlock) k_bin_scatter(PGrid c, int64_t np, const float* __restrict__ pos,
                                                        uint32_t* cursor, uint32_t* __restrict__ order,
                                                        float* __restrict__ pos_s, const float* __restrict__ vel,
                                                        float* __restrict__ vel_s) {
    const int64_t p = int64_t(xcd_block()) * kBlock + threadIdx.x;
    if (p >= np) return;
    const float px = pos[3 * p], py = pos[3 * p + 1], pz = pos[3 * p + 2];
    const uint32_t slot = atomicAdd(&cursor[bin_of(c, px, py, pz)], 1u);
    order[slot] = uint32_t(p);
    pos_s[3 * size_t(slot)] = px;
    pos_s[3 * size_t(slot) + 1] = py;
    pos_s[3 * size_t(slot) + 2] = pz;
    if (vel) {
        vel_s[3 * size_t(slot)] = vel[3 * p];
        vel_s[3 * size_t(slot) + 1] = vel[3 * p + 1];
        vel_s[3 * size_t(slot) + 2] = vel[3 * p + 2];
    }
}

// Two passes per target grid (the cells, or the faces of one axis; LINEAR
// kernel).  Pass 1, one work-item per bin: every particle of the bin adds
// its weights, and weight times value, to slots indexed by the target node
// relative to the bin's first node clamp(s) (two slots per axis, three on the
// axis the target grid is shifted along: its support starts at the cell
// grid's corner or the next).  A support's corners that clamp onto one node
// share a slot, so an edge bin collects far-outside particles too.  Empty
// bins write nothing.  Pass 2, one work-item per node: the sum, in a fixed bin
// order, of the slots of the non-empty neighbouring bins that point at it;
// then the normalisation.
constexpr int kSlotsMax = 12;

__device__ __forceinline__ int clamp_bin(int s, int cells) { return s < -1 ? -1 : (s > cells - 1 ? cells - 1 : s); }

// pos_s: positions in bin order; val is in bin order too when val_sorted,
// else indexed by particle through order.
template <int SHIFT>
__global__ void __launch_bounds__(kBlock) k_p2g_bins(PGrid g, BinGrid bg, const uint32_t* __restrict__ start,
                                                     const uint32_t* __restrict__ order, const float* __restrict__ pos_s,
                                                     const float* __restrict__ val, int span, int off, int val_sorted,
                                                     float* __restrict__ acc) {
    const size_t nb = size_t(bg.nx + 1) * (bg.ny + 1) * (bg.nz + 1);
    const size_t b = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (b >= nb) return;
    const int s[3] = {int(b % uint32_t(bg.nx + 1)) - 1, int((b / uint32_t(bg.nx + 1)) % uint32_t(bg.ny + 1)) - 1,
                      int(b / (size_t(bg.nx + 1) * uint32_t(bg.ny + 1))) - 1};
    const int len[3] = {g.nx, g.ny, g.nz};
    constexpr int ns[3] = {SHIFT == 0 ? 3 : 2, SHIFT == 1 ? 3 : 2, SHIFT == 2 ? 3 : 2};
    int base[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) base[a] = clampi(s[a], len[a]);
    const uint32_t q0 = start[b], q1 = start[b + 1];
    if (q0 == q1) return;   // an empty bin's slots are never read
    float sv[kSlotsMax], sw[kSlotsMax];
#pragma unroll
    for (int q = 0; q < kSlotsMax; ++q) sv[q] = sw[q] = 0.0f;
    for (uint32_t q = q0; q < q1; ++q) {
        PStencil st;
        pg_stencil(g, pos_s[3 * size_t(q)], pos_s[3 * size_t(q) + 1], pos_s[3 * size_t(q) + 2], MGF_PG_LINEAR, st);
        const float v = val[size_t(span) * (val_sorted ? q : order[q]) + off];
        // per-axis slot weights: the corners that clamp onto slot t
        float W[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int t = 0; t < 3; ++t) W[a][t] = 0.0f;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int t = clampi(st.i0[a] + c, len[a]) - base[a];
#pragma unroll
                for (int u = 0; u < 3; ++u)
                    if (t == u) W[a][u] += st.w[a][c];
            }
        }
#pragma unroll
        for (int tz = 0; tz < ns[2]; ++tz)
#pragma unroll
            for (int ty = 0; ty < ns[1]; ++ty)
#pragma unroll
                for (int tx = 0; tx < ns[0]; ++tx) {
                    const int slot = (tz * ns[1] + ty) * ns[0] + tx;
                    const float wt = W[0][tx] * W[1][ty] * W[2][tz];
                    sv[slot] += wt * v;
                    sw[slot] += wt;
                }
    }
    constexpr int nslot = ns[0] * ns[1] * ns[2];
#pragma unroll
    for (int u = 0; u < kSlotsMax; ++u)
        if (u < nslot) {
            acc[(2 * size_t(u)) * nb + b] = sv[u];
            acc[(2 * size_t(u) + 1) * nb + b] = sw[u];
        }
}

__global__ void __launch_bounds__(kBlock) k_p2g_nodes(PGrid g, int shift, BinGrid bg, const uint32_t* __restrict__ start,
                                                      const float* __restrict__ acc, float* __restrict__ field,
                                                      float* __restrict__ weight, int normalize) {
    const size_t total = size_t(g.nx) * g.ny * g.nz;
    const size_t node = size_t(xcd_block()) * kBlock + threadIdx.x;
    if (node >= total) return;
    const size_t nb = size_t(bg.nx + 1) * (bg.ny + 1) * (bg.nz + 1);
    const int idx[3] = {int(node % uint32_t(g.nx)), int((node / uint32_t(g.nx)) % uint32_t(g.ny)),
                        int(node / (size_t(g.nx) * uint32_t(g.ny)))};
    const int len[3] = {g.nx, g.ny, g.nz}, cells[3] = {bg.nx, bg.ny, bg.nz};
    int ns[3], s0[3], s1[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        ns[a] = a == shift ? 3 : 2;
        s0[a] = clamp_bin(idx[a] - ns[a], cells[a]);
        s1[a] = clamp_bin(idx[a], cells[a]);
    }
    float sv = 0.0f, sw = 0.0f;
    for (int bz = s0[2]; bz <= s1[2]; ++bz) {
        const int tz = idx[2] - clampi(bz, len[2]);
        if (tz < 0 || tz >= ns[2]) continue;
        for (int by = s0[1]; by <= s1[1]; ++by) {
            const int ty = idx[1] - clampi(by, len[1]);
            if (ty < 0 || ty >= ns[1]) continue;
            for (int bx = s0[0]; bx <= s1[0]; ++bx) {
                const int tx = idx[0] - clampi(bx, len[0]);
                if (tx < 0 || tx >= ns[0]) continue;
                const size_t b = (size_t(bz + 1) * uint32_t(bg.ny + 1) + uint32_t(by + 1)) * uint32_t(bg.nx + 1) +
                                 uint32_t(bx + 1);
                if (start[b] == start[b + 1]) continue;   // empty bin: no slots written
                const size_t slot = size_t((tz * ns[1] + ty) * ns[0] + tx);
                sv += acc[2 * slot * nb + b];
                sw += acc[(2 * slot + 1) * nb + b];
            }
        }
    }
    field[node] = normalize && sw > 0.0f ? sv / sw : sv;
    weight[node] = sw;
}

// ===========================================================================
static PGrid pgrid_of(const GridDev& g, int kind) {
    PGrid p{g.nx, g.ny, g.nz, g.ox, g.oy, g.oz, g.hx, g.hy, g.hz, g.rhx, g.rhy, g.rhz, g.pow2};
    if (kind == 1) { p.nx += 1; p.ox = g.ox - g.hx / 2; }
    if (kind == 2) { p.ny += 1; p.oy = g.oy - g.hy / 2; }
    if (kind == 3) { p.nz += 1; p.oz = g.oz - g.hz / 2; }
    return p;
}

size_t pg_field_count(const GridDev& g, int kind) {
    const PGrid p = pgrid_of(g, kind);
    return size_t(p.nx) * p.ny * p.nz;
}

// Scratch of launch_p2g: counters, prefix and cursor a tile, the chunks, and
// the order of one segment's particles.
static size_t splat_tile_cap(const GridDev& g) {
    return size_t(splat_tiles(g.nx + 1, 4)) * splat_tiles(g.ny + 1, 4) * splat_tiles(g.nz + 1, 4);
}
static size_t splat_work_cap(size_t nt, size_t seg) { return std::min(nt, seg) + seg / kSplatChunk + 1; }

// Whether the splat sorts (else k_p2g_hash), by what either costs: the sort a
// little for every tile (the scan) and more for each that holds particles (an
// LDS tile to clear and flush), the hash table a constant (its chain of probes)
// and more for each particle.  The constants are in ns, from particles spread
// over whole grids, hash / sort in us:
//   64^3 cells    100: LINEAR 39 / 34, QUADRATIC 214 / 36, CUBIC 215 / 41
//   256^3 (36K tiles)
//     LINEAR      100 50 / 99, 100K 125 / 270, 300K 285 / 295, 1M 824 / 439
//     QUADRATIC   100 228 / 106, 10K 260 / 287, 100K 668 / 592, 1M 6230 / 773
//     CUBIC       100 230 / 106, 10K 260 / 506, 100K 669 / 1500, 300K 1950 / 1760
//   512^3 (275K)  LINEAR 1M 1010 / 1940, 3M 2500 / 2170; QUADRATIC 300K 2130 / 3210,
//                 1M 6430 / 4620; CUBIC 1M 6420 / 12100, 3M 18600 / 13800
// Sets that fill a part of the grid have fewer tiles with particles than is
// assumed, so grids whose tiles fit the window sort the wide kernels at any
// count (10K CUBIC in 0.3 of 160 x 160 x 117, three fields each way: 815 / 524; the
// same spread over 160^3 would be some 0.1 ms a field slower than the table).
// P2GSUM adds one value a particle and little is left to save: 300K over 64^3
// cells 36 / 51, 1M 72 / 72, 1M over 32^3 131 / 66; 5.0M moved by up to 4 cells
// against their order 333 / 135, but in order 76 / 106; beyond the window 40M
// moved 1940 / 1130, in order 454 / 840, 8M in random order 442 / 1196.
static bool splat_sorts(const GridDev& g, int64_t np, int alg) {
    if (np <= 0) return false;
    const double nt = double(splat_tile_cap(g)), n = double(np), held = std::min(n, nt);
    switch (alg) {
        case MGF_PG_P2GSUM: return n >= 786432.0 && nt <= double(kSplatLdsTiles);
        case MGF_PG_LINEAR: return 1.4 * nt + 6.0 * held <= 12.0e3 + 0.74 * n;
        case MGF_PG_QUADRATIC: return nt <= double(kSplatLdsTiles) || 1.4 * nt + 18.0 * held <= 170.0e3 + 6.0 * n;
        default: return nt <= double(kSplatLdsTiles) || 1.4 * nt + 41.0 * held <= 170.0e3 + 6.0 * n;
    }
}

size_t p2g_work_words(const GridDev& g, int64_t np, int alg) {
    if (!splat_sorts(g, np, alg)) return 0;
    const size_t nt = splat_tile_cap(g), seg = size_t(std::min<int64_t>(std::max<int64_t>(np, 1), kSplatSegment));
    return 3 * nt + 2 + 2 * splat_work_cap(nt, seg) + seg;
}

template <int ALG>
static hipError_t splat_segment(hipStream_t s, const PGrid& p, uint32_t np, const float* pos, const float* val, int span,
                                int off, uint32_t* work, size_t cap, float* field, float* weight) {
    constexpr int N = splat_corners(ALG);
    const size_t nt = size_t(splat_tiles(p.nx, N)) * splat_tiles(p.ny, N) * splat_tiles(p.nz, N);
    const size_t nw = splat_work_cap(nt, np);
    uint32_t *counts = work, *start = counts + cap, *cursor = start + cap + 1, *nwork = cursor + cap,
             *list = nwork + 1, *order = list + 2 * splat_work_cap(cap, np);
    const uint32_t lds = uint32_t(std::min<size_t>(nt, kSplatLdsTiles));
    const dim3 sg((np + kBlock * kSplatItems - 1) / (kBlock * kSplatItems));
    hipError_t e = launch_dims(k_splat_count<ALG>, "k_splat_count", sg, dim3(kBlock), lds * 4u, s, p, np, pos, counts,
                               uint32_t(nt));
    if (e != hipSuccess) return e;
    e = launch_dims(k_splat_scan, "k_splat_scan", dim3(1), dim3(1024), 0, s, uint32_t(nt), counts, start, cursor, list,
                    nwork);
    if (e == hipSuccess)
        e = launch_dims(k_splat_order<ALG>, "k_splat_order", sg, dim3(kBlock), lds * 4u, s, p, np, pos, cursor, order,
                        uint32_t(nt));
    if (e == hipSuccess)
        e = launch_dims(k_splat_tiles<ALG>, "k_splat_tiles", dim3(uint32_t(nw)), dim3(kSplatBlock), 0, s, p, pos, val,
                        span, off, start, order, list, nwork, field, weight);
    return e;
}

template <int ALG>
static hipError_t splat_hash(hipStream_t s, const PGrid& p, int64_t np, const float* pos, const float* val, int span,
                             int off, float* field, float* weight) {
    return LAUNCH(k_p2g_hash<ALG>, grid_for(size_t(np)), p, np, pos, val, span, off, field, weight);
}

hipError_t launch_p2g(hipStream_t s, const GridDev& g, int kind, int64_t np, const float* pos, const float* val,
                      int span, int off, int alg, float* field, float* weight, int normalize, uint32_t* work) {
    const PGrid p = pgrid_of(g, kind);
    const size_t n = size_t(p.nx) * p.ny * p.nz, cap = splat_tile_cap(g);
    const bool sorted = work && splat_sorts(g, np, alg);
    hipError_t e = hipSuccess;
    int64_t first = 0;
    do {
        // counts of a segment; the field and the weight once
        const size_t nf = first ? 0 : n, nc = sorted ? cap : 0;
        e = LAUNCH(k_splat_clear, grid_for(std::max(nf, nc)), nf, field, weight, nc, work);
        const int64_t m = sorted ? std::min<int64_t>(np - first, kSplatSegment) : np;
        if (e != hipSuccess || m <= 0) break;
        const float* ps = pos + 3 * first;
        const float* vs = val + int64_t(span) * first;
        auto run = [&](auto a) {
            constexpr int ALG = decltype(a)::value;
            return sorted ? splat_segment<ALG>(s, p, uint32_t(m), ps, vs, span, off, work, cap, field, weight)
                          : splat_hash<ALG>(s, p, m, ps, vs, span, off, field, weight);
        };
        switch (alg) {
            case MGF_PG_P2GSUM: e = run(std::integral_constant<int, MGF_PG_P2GSUM>()); break;
            case MGF_PG_LINEAR: e = run(std::integral_constant<int, MGF_PG_LINEAR>()); break;
            case MGF_PG_QUADRATIC: e = run(std::integral_constant<int, MGF_PG_QUADRATIC>()); break;
            default: e = run(std::integral_constant<int, MGF_PG_CUBIC>()); break;
        }
        first += m;
    } while (e == hipSuccess && first < np);
    if (e == hipSuccess && normalize) e = LAUNCH(k_p2g_normalize, grid_for(n), n, field, weight);
    return e;
}

hipError_t launch_g2p(hipStream_t s, const GridDev& g, int kind, int64_t np, const float* pos, const float* field,
                      int alg, float* val, int span, int off) {
    if (np <= 0) return hipSuccess;
    if (alg == MGF_PG_QUADRATIC || alg == MGF_PG_CUBIC)
        return LAUNCH(k_g2p<4>, grid_for(size_t(np)), pgrid_of(g, kind), np, pos, field, alg, val, span, off);
    return LAUNCH(k_g2p<2>, grid_for(size_t(np)), pgrid_of(g, kind), np, pos, field, alg, val, span, off);
}

hipError_t launch_particle_markers(hipStream_t s, const GridDev& g, const float* solid, int64_t np, const float* pos,
                                   float* out) {
    const size_t n = size_t(g.nx) * g.ny * g.nz;
    hipError_t e = launch_fill(s, out, n, 0.0f);
    if (e == hipSuccess && np > 0) e = LAUNCH(k_particle_counts, grid_for(size_t(np)), pgrid_of(g, 0), np, pos, out);
    if (e == hipSuccess && solid) e = LAUNCH(k_particle_markers, grid_for(n), n, solid, out);
    return e;
}

hipError_t launch_axpy_n(hipStream_t s, size_t n, float a, const float* x, float* y) {
    if (n == 0) return hipSuccess;
    return LAUNCH(k_axpy_n, grid_for(n), n, a, x, y);
}

hipError_t launch_scale_n(hipStream_t s, size_t n, float a, float* x) {
    if (n == 0) return hipSuccess;
    return LAUNCH(k_scale_n, grid_for(n), n, a, x);
}

hipError_t launch_clamp_particles(hipStream_t s, const GridDev& g, int64_t np, float* pos) {
    const int64_t m = std::min<int64_t>(np, int64_t(g.nx) * g.ny * g.nz);
    if (m <= 0) return hipSuccess;
    const float hx = g.ox + float(g.nx) * g.hx, hy = g.oy + float(g.ny) * g.hy, hz = g.oz + float(g.nz) * g.hz;
    return LAUNCH(k_clamp_particles, grid_for(size_t(m)), m, pos, g.ox, g.oy, g.oz, hx, hy, hz);
}

}  // namespace mgf

namespace mgf {

uint32_t gen_tiles(size_t ncell) { return uint32_t((ncell + kGenTile - 1) / kGenTile); }

hipError_t launch_gen_count(hipStream_t s, size_t ncell, const float* fluid, const float* solid, uint32_t* tiles) {
    const uint32_t nt = gen_tiles(ncell);
    (void)launch_dims(k_gen_count, "k_gen_count", dim3(nt), dim3(kBlock), 0, s, ncell, fluid, solid, tiles);
    (void)launch_dims(k_gen_scan, "k_gen_scan", dim3(1), dim3(1024), 0, s, nt, tiles);
    return hipGetLastError();
}

hipError_t launch_gen_emit(hipStream_t s, const GridDev& g, const float* fluid, const float* solid,
                           const uint32_t* tiles, int per_cell, uint64_t seed, float* pos) {
    const size_t ncell = size_t(g.nx) * g.ny * g.nz;
    (void)launch_dims(k_gen_emit, "k_gen_emit", dim3(gen_tiles(ncell)), dim3(kBlock), 0, s, g, ncell, fluid, solid, tiles,
                       per_cell, seed, pos);
    return hipGetLastError();
}

hipError_t launch_flip_delta(hipStream_t s, size_t n, const float* in, float* delta) {
    if (n == 0) return hipSuccess;
    return LAUNCH(k_flip_delta, grid_for(n), n, in, delta);
}

hipError_t launch_particle_markers_u8(hipStream_t s, const GridDev& g, const uint8_t* solid_mask, int64_t np,
                                      const float* pos, uint8_t* markers) {
    const size_t n = size_t(g.nx) * g.ny * g.nz;
    hipError_t e = LAUNCH(k_markers_solid, grid_for(n), n, solid_mask, markers);
    if (e == hipSuccess && np > 0)
        e = LAUNCH(k_markers_particles, grid_for(size_t(np)), pgrid_of(g, 0), np, pos, markers);
    return e;
}

}  // namespace mgf

namespace mgf {

// Work-groups of the kernels that reduce a maximum: a multiple of the XCD
// count, a few per CU, each looping over its share.
constexpr uint32_t kMaxReduceBlocks = 4096;

hipError_t launch_transfer_vel(hipStream_t s, const GridDev& g, int64_t np, const float* pos,
                               const float* const in[3], const float* const delta[3], int kind, int alg, float keep,
                               float mixing, float* vel) {
    if (np <= 0) return hipSuccess;
    const Faces3 fi{{in[0], in[1], in[2]}};
    const Faces3 fd{{delta ? delta[0] : nullptr, delta ? delta[1] : nullptr, delta ? delta[2] : nullptr}};
    if (alg == MGF_PG_QUADRATIC || alg == MGF_PG_CUBIC)
        return LAUNCH(k_transfer_vel<4>, grid_for(size_t(np)), pgrid_of(g, 1), pgrid_of(g, 2), pgrid_of(g, 3), np,
                      pos, fi, fd, kind, alg, keep, mixing, vel);
    return LAUNCH(k_transfer_vel<2>, grid_for(size_t(np)), pgrid_of(g, 1), pgrid_of(g, 2), pgrid_of(g, 3), np, pos,
                  fi, fd, kind, alg, keep, mixing, vel);
}

hipError_t launch_sample_absmax(hipStream_t s, const GridDev& g, Vel V, int64_t np, const float* pos, float* out,
                                uint32_t* vmax_bits) {
    hipError_t e = hipMemsetAsync(vmax_bits, 0, sizeof(uint32_t), s);
    if (e != hipSuccess || np <= 0) return e;
    return LAUNCH(k_sample_absmax, std::min<uint32_t>(grid_for(size_t(np)), kMaxReduceBlocks), g, V, np, pos, out,
                  vmax_bits);
}

hipError_t launch_rk_substep(hipStream_t s, const GridDev& g, Vel V, int64_t np, float* pos, float* v1, int order,
                             float step, float half, float three_q, float c1, float c2, float c3, int resample,
                             uint32_t* vmax_bits) {
    hipError_t e = hipSuccess;
    if (resample) e = hipMemsetAsync(vmax_bits, 0, sizeof(uint32_t), s);
    if (e != hipSuccess || np <= 0) return e;
    return LAUNCH(k_rk_substep, std::min<uint32_t>(grid_for(size_t(np)), kMaxReduceBlocks), g, V, np, pos, v1, order,
                  step, half, three_q, c1, c2, c3, resample, vmax_bits);
}

}  // namespace mgf

namespace mgf {

size_t bin_count(const GridDev& g) { return size_t(g.nx + 1) * size_t(g.ny + 1) * size_t(g.nz + 1); }
uint32_t bin_tiles(const GridDev& g) { return gen_tiles(bin_count(g)); }

hipError_t launch_bin_particles(hipStream_t s, const GridDev& g, int64_t np, const float* pos, uint32_t* counts,
                                uint32_t* tiles, uint32_t* start, uint32_t* cursor, uint32_t* order, float* pos_s,
                                const float* vel, float* vel_s) {
    const size_t nb = bin_count(g);
    const uint32_t nt = gen_tiles(nb);
    const PGrid c = pgrid_of(g, 0);
    hipError_t e = hipMemsetAsync(counts, 0, nb * sizeof(uint32_t), s);
    if (e == hipSuccess && np > 0) e = LAUNCH(k_bin_count, grid_for(size_t(np)), c, np, pos, counts);
    if (e != hipSuccess) return e;
    (void)launch_dims(k_scan_tiles, "k_scan_tiles", dim3(nt), dim3(kBlock), 0, s, nb, counts, tiles);
    (void)launch_dims(k_gen_scan, "k_gen_scan", dim3(1), dim3(1024), 0, s, nt, tiles);
    (void)launch_dims(k_scan_apply, "k_scan_apply", dim3(nt), dim3(kBlock), 0, s, nb, counts, tiles, nt, start, cursor);
    e = hipGetLastError();
    if (e == hipSuccess && np > 0)
        e = LAUNCH(k_bin_scatter, grid_for(size_t(np)), c, np, pos, cursor, order, pos_s, vel, vel_s);
    return e;
}

size_t p2g_acc_floats(const GridDev& g) { return 2 * size_t(kSlotsMax) * bin_count(g); }

hipError_t launch_p2g_binned(hipStream_t s, const GridDev& g, int kind, const uint32_t* start, const uint32_t* order,
                             const float* pos_s, const float* val, int span, int off, int val_sorted, float* acc,
                             float* field, float* weight, int normalize) {
    const PGrid p = pgrid_of(g, kind);
    const size_t n = size_t(p.nx) * p.ny * p.nz;
    const BinGrid bg{g.nx, g.ny, g.nz};
    const uint32_t gb = grid_for(bin_count(g));
    hipError_t e;
    switch (kind) {
        case 1: e = LAUNCH(k_p2g_bins<0>, gb, p, bg, start, order, pos_s, val, span, off, val_sorted, acc); break;
        case 2: e = LAUNCH(k_p2g_bins<1>, gb, p, bg, start, order, pos_s, val, span, off, val_sorted, acc); break;
        case 3: e = LAUNCH(k_p2g_bins<2>, gb, p, bg, start, order, pos_s, val, span, off, val_sorted, acc); break;
        default: e = LAUNCH(k_p2g_bins<-1>, gb, p, bg, start, order, pos_s, val, span, off, val_sorted, acc); break;
    }
    if (e == hipSuccess) e = LAUNCH(k_p2g_nodes, grid_for(n), p, kind - 1, bg, start, acc, field, weight, normalize);
    return e;
}

}  // namespace mgf
