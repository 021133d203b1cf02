// flip_kernels.hpp -- gfx950 kernels of the FLIP substep (included once, by flip_solver.hip).
// Each kernel is a functor launched through k_one / k_many (flip_launch.hpp).
//
// Layout in HBM (one scene):
//   particles   SoA float px..vz, grid coordinates gx..gz, uint32 id; kept cell-sorted after binning
//   MAC faces   u (nx+1,ny,nz), v (nx,ny+1,nz), w (nx,ny,nz+1), x-fastest (Array.h:276)
//   cells       phi (nx,ny,nz) float; cell_start (nx*ny*nz + 1) uint32
//   pressure    8^3-cell bricks holding >= 1 fluid cell, 512 cells contiguous per brick
//               (brick-major, x-fastest inside a brick): vectors, matrix diagonal and the three
//               "upper" couplings (+x,+y,+z); a brick's 6 neighbours come from a slot table.
#pragma once

#include "flip_device.hpp"
#include "flip_launch.hpp"

namespace bnn {

constexpr int kBlock = 256;

//==================================================================================================
// moveParticles: RK2 through the grid + domain-box projection (PIC_Solver.cpp:353-373, 1137-1144;
// BoundaryObject.cpp:72-90)
//==================================================================================================
struct VelGrid {
    const float *u, *v, *w;
};

// APIC / AFLIP affine matrices, nine arrays in the particles' storage order: c[3 d + e] = C_d[e]
struct Affine {
    float* c[9];
};

__device__ __forceinline__ void vel_from_grid(const VelGrid& G, const GridGeom& g, float gpx, float gpy, float gpz, float& ux,
                                              float& uy, float& uz) {
    ux = interp3(G.u, g.nx + 1, g.ny, g.nz, gpx, gpy - 0.5f, gpz - 0.5f);
    uy = interp3(G.v, g.nx, g.ny + 1, g.nz, gpx - 0.5f, gpy, gpz - 0.5f);
    uz = interp3(G.w, g.nx, g.ny, g.nz + 1, gpx - 0.5f, gpy - 0.5f, gpz);
}

//==================================================================================================
// Binning: stable counting sort by linear cell index (Grid.cpp:92-114, 283-309)
//==================================================================================================
__device__ __forceinline__ int cell_axis(float p, float bmin, float dx, int n) {
    int c = (int)((p - bmin) / dx);  // Grid.h:156-162 (truncation toward zero)
    return c < 0 ? 0 : (c > n - 1 ? n - 1 : c);  // Grid::getValidCellIdx clamp
}

// Runs of equal keys inside a wavefront (particles arrive almost cell-sorted from the previous
// substep, so a run usually covers a whole cell): the run's first lane does one atomic for the run.
// Returns the run length in the leader lane, 0 elsewhere; `leader` gets the run's first lane.
__device__ __forceinline__ uint32_t key_run(uint32_t c, bool active, int& leader) {
    const int      lane  = (int)(threadIdx.x & 63);
    const uint32_t prev  = __shfl_up(c, 1, 64);
    const bool     first = active && (lane == 0 || prev != c);
    const uint64_t heads = __ballot(first);
    const uint64_t live  = __ballot(active);
    const uint64_t upTo  = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
    leader               = 63 - __clzll(heads & upTo);
    if(!first) return 0u;
    const uint64_t after = heads & ~upTo;           // later run heads
    const int      end   = after ? __ffsll((unsigned long long)after) - 1 : 64 - __clzll(live);
    return (uint32_t)(end - lane);
}

// A particle's cell: its key, the cell's count and the occupancy of its brick. Called by whole wavefronts.
struct CellKeys {
    uint32_t* key;
    uint32_t* count;
    uint8_t*  occ;  // per 8^3 cell brick: 1 when a particle lies in it (cleared before)
    __device__ __forceinline__ void put(const GridGeom& g, uint32_t p, bool active, float x, float y, float z) const {
        uint32_t c = 0xFFFFFFFFu, brick = 0;
        if(active) {
            const int i = cell_axis(x, g.bminx, g.dx, g.nx);
            const int j = cell_axis(y, g.bminy, g.dx, g.ny);
            const int k = cell_axis(z, g.bminz, g.dx, g.nz);
            c           = (uint32_t)lin3(i, j, k, g.nx, g.ny);
            brick       = (uint32_t)(((k >> 3) * g.nby + (j >> 3)) * g.nbx + (i >> 3));
            key[p]      = c;
        }
        int            leader;
        const uint32_t len = key_run(c, active, leader);
        if(len) {
            atomicAdd(&count[c], len);
            occ[brick] = 1;
        }
    }
};

// out.key set: the binning that follows at once takes its keys from here, where the new position is in
// registers, instead of reading it back: k_cell_key took 158 us at 256^3, the move is bound by its gathers
// and hides most of that (the step 13.74 -> 13.61 ms, a 128^3 frame 16.5 -> 16.3).
struct k_move {
    static constexpr int kThreads = kBlock;
    static constexpr bool kByAddress = true;
    Particles P;
    uint32_t n;
    VelGrid G;
    GridGeom g;
    BndSet bnd;
    float dt;
    uint32_t advSteps;
    int reflect;
    float reflMult;
    CellKeys out;
    __device__ void operator()(Blk blk) const {
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        float x = 0.f, y = 0.f, z = 0.f;
        if(p < n) move(p, x, y, z);
        if(out.key) out.put(g, p, p < n, x, y, z);
    }
    __device__ __forceinline__ void move(uint32_t p, float& x, float& y, float& z) const {
        x = P.px[p];
        y = P.py[p];
        z = P.pz[p];
        float vx = P.vx[p], vy = P.vy[p], vz = P.vz[p];
        bool  changed = false;
        const float sub = dt / (float)advSteps;
        for(uint32_t s = 0; s < advSteps; ++s) {
            // trace_rk2
            float ux, uy, uz;
            vel_from_grid(G, g, (x - g.bminx) / g.dx, (y - g.bminy) / g.dx, (z - g.bminz) / g.dx, ux, uy, uz);
            const float h  = 0.5f * sub;
            const float mx = x + h * ux, my = y + h * uy, mz = z + h * uz;
            vel_from_grid(G, g, (mx - g.bminx) / g.dx, (my - g.bminy) / g.dx, (mz - g.bminz) / g.dx, ux, uy, uz);
            x = x + sub * ux;
            y = y + sub * uy;
            z = z + sub * uz;
            // constrainToBoundary(ppos, pvel) of every boundary object
            if(bnd_constrain(bnd, x, y, z, vx, vy, vz, reflect, reflMult)) changed = true;
        }
        P.px[p] = x;
        P.py[p] = y;
        P.pz[p] = z;
        if(changed) {
            P.vx[p] = vx;
            P.vy[p] = vy;
            P.vz[p] = vz;
        }
    }
};

// (i, j, k) of the linear index t of an sx x sy x sz array (x fastest), in 32-bit arithmetic: every
// grid array here has fewer than 2^32 entries, and 64-bit division is many instructions on the GPU
__device__ __forceinline__ void unlin3(uint32_t t, int sx, int sy, int& i, int& j, int& k) {
    const uint32_t r = t / (uint32_t)sx;
    i                = (int)(t - r * (uint32_t)sx);
    j                = (int)(r % (uint32_t)sy);
    k                = (int)(r / (uint32_t)sy);
}

struct k_cell_key {
    static constexpr int kThreads = kBlock;
    const float* __restrict__ px;
    const float* __restrict__ py;
    const float* __restrict__ pz;
    uint32_t n;
    GridGeom g;
    CellKeys out;
    __device__ void operator()(Blk blk) const {
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        const bool     active = p < n;
        out.put(g, p, active, active ? px[p] : 0.f, active ? py[p] : 0.f, active ? pz[p] : 0.f);
    }
};

// counts return to zero here (each particle takes one slot), so the count array needs no clearing;
// a run's lanes take consecutive slots in lane order
struct k_scatter {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ key;
    uint32_t n;
    const uint32_t* __restrict__ cell_start;
    uint32_t* __restrict__ count;
    uint32_t* __restrict__ perm;
    __device__ void operator()(Blk blk) const {
        const uint32_t p      = blk.id * blockDim.x + threadIdx.x;
        const bool     active = p < n;
        const uint32_t c      = active ? key[p] : 0xFFFFFFFFu;
        int            leader;
        const uint32_t len  = key_run(c, active, leader);
        uint32_t       left = 0;  // count before the run's subtraction
        if(len) left = atomicSub(&count[c], len);
        left = __shfl(left, leader, 64);
        const uint32_t runLen = __shfl(len, leader, 64);
        if(active) perm[cell_start[c] + left - runLen + (uint32_t)((int)(threadIdx.x & 63) - leader)] = p;
    }
};

// make each cell's segment ascending: the counting sort becomes stable (ties by particle index)
struct k_segsort {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ cell_start;
    uint32_t ncells;
    uint32_t* __restrict__ perm;
    __device__ void operator()(Blk blk) const {
        const uint32_t c = blk.id * blockDim.x + threadIdx.x;
        if(c >= ncells) return;
        const uint32_t b = cell_start[c], e = cell_start[c + 1];
        if(e - b < 2) return;
        if(e - b <= 16) {
            // up to 16 entries in registers (padding sorts to the end): most cells arrive in order and
            // are left as they are; the others are sorted by odd-even transposition (the entries are
            // distinct particle indices, so the order is the one the insertion sort below gives)
            const uint32_t n = e - b;
            uint32_t       r[16];
#pragma unroll
            for(uint32_t k = 0; k < 16; ++k) r[k] = k < n ? perm[b + k] : 0xFFFFFFFFu;
            bool sorted = true;
#pragma unroll
            for(uint32_t k = 1; k < 16; ++k) sorted &= r[k - 1] <= r[k];
            if(sorted) return;
#pragma unroll
            for(int ph = 0; ph < 16; ++ph) {
#pragma unroll
                for(int k = ph & 1; k + 1 < 16; k += 2) {
                    const uint32_t lo = min(r[k], r[k + 1]), hi = max(r[k], r[k + 1]);
                    r[k]              = lo;
                    r[k + 1]          = hi;
                }
            }
#pragma unroll
            for(uint32_t k = 0; k < 16; ++k)
                if(k < n) perm[b + k] = r[k];
            return;
        }
        for(uint32_t i = b + 1; i < e; ++i) {
            uint32_t v = perm[i];
            uint32_t j = i;
            while(j > b && perm[j - 1] > v) {
                perm[j] = perm[j - 1];
                --j;
            }
            perm[j] = v;
        }
    }
};

struct k_permute {
    static constexpr int kThreads = kBlock;
    Particles in;
    Particles out;
    const uint32_t* __restrict__ perm;
    uint32_t n;
    GridGeom g;
    __device__ void operator()(Blk blk) const {
        const uint32_t i = blk.id * blockDim.x + threadIdx.x;
        if(i >= n) return;
        const uint32_t s = perm[i];
        const float    x = in.px[s], y = in.py[s], z = in.pz[s];
        const float    vx = in.vx[s], vy = in.vy[s], vz = in.vz[s];
        out.px[i]        = x;
        out.py[i]        = y;
        out.pz[i]        = z;
        out.vx[i]        = vx;
        out.vy[i]        = vy;
        out.vz[i]        = vz;
        out.id[i]        = in.id[s];
        out.gp[i]        = make_float4((x - g.bminx) / g.dx, (y - g.bminy) / g.dx, (z - g.bminz) / g.dx, vx);
        out.gv[i]        = make_float2(vy, vz);
    }
};

// the velocities' copy in gp.w / gv refreshed from the velocity arrays (particles already binned)
struct k_pack_velocity {
    static constexpr int kThreads = kBlock;
    Particles P;
    uint32_t n;
    __device__ void operator()(Blk blk) const {
        const uint32_t i = blk.id * blockDim.x + threadIdx.x;
        if(i >= n) return;
        P.gp[i].w = P.vx[i];
        P.gv[i]   = make_float2(P.vy[i], P.vz[i]);
    }
};

// three particle arrays as triples in the caller's order, for readback: out[3 id + d]. A host loop over six
// copied arrays did this before: a z-sort and readback of 1.7M particles took 11.7 ms, 1.0 now; a frame of
// five substeps and readback of 4M 55.3, 20.4 now (both end in the copy over PCIe, about 53 GB/s).
struct k_user_order {
    static constexpr int kThreads = kBlock;
    const float* __restrict__ x;
    const float* __restrict__ y;
    const float* __restrict__ z;
    const uint32_t* __restrict__ id;
    uint32_t n;
    float* __restrict__ out;
    __device__ void operator()(Blk blk) const {
        const uint32_t i = blk.id * blockDim.x + threadIdx.x;
        if(i >= n) return;
        float* o = out + 3 * (size_t)id[i];
        o[0] = x[i];
        o[1] = y[i];
        o[2] = z[i];
    }
};

//==================================================================================================
// Z-order sort of the particles (PIC_Solver.cpp:315-328 -> NeighborSearch::z_sort,
// NeighborSearch.cpp:45-86). Keys are built in the caller's particle order; a stable LSD radix sort
// on 8-bit digits gives the permutation; the particles' external ids are renamed by it (storage on
// the device stays cell-sorted, so no particle data moves).
//==================================================================================================
// NeighborSearch::cell_index (NeighborSearch.cpp:47-55) and the shift of z_value (:60-70): cell of
// x - 1.2345 through the reciprocal cell size (floor for negative offsets), then minus (INT_MIN + 1).
__device__ __forceinline__ uint64_t zsort_coord(float x, float inv) {
    const float tmp = x - 1.2345f;
    const int   k   = tmp >= 0.f ? (int)(inv * tmp) : (int)(inv * tmp) - 1;
    return (uint64_t)((int64_t)k + 2147483647ll);
}
// bit b of v (b < 21) to bit 3b
__device__ __forceinline__ uint64_t spread_by_3(uint64_t v) {
    v &= 0x1FFFFFull;
    v = (v | v << 32) & 0x001F00000000FFFFull;
    v = (v | v << 16) & 0x001F0000FF0000FFull;
    v = (v | v << 8) & 0x100F00F00F00F00Full;
    v = (v | v << 4) & 0x10C30C30C30C30C3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}
// morton3D_64_encode (Morton3D.h:54-66) keeps, in 64 bits, bit b of coordinate d at bit 3b + d:
// 22 bits of x, 21 of y and z.
__device__ __forceinline__ uint64_t zsort_key(float x, float y, float z, float inv) {
    const uint64_t cx = zsort_coord(x, inv), cy = zsort_coord(y, inv), cz = zsort_coord(z, inv);
    return spread_by_3(cx) | spread_by_3(cy) << 1 | spread_by_3(cz) << 2 | ((cx >> 21) & 1ull) << 63;
}

// keys in external order, split in 32-bit halves; values = external index
struct k_zsort_keys {
    static constexpr int kThreads = kBlock;
    Particles P;
    uint32_t n;
    float inv;
    uint32_t* __restrict__ klo;
    uint32_t* __restrict__ khi;
    uint32_t* __restrict__ val;
    __device__ void operator()(Blk blk) const {
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        if(p >= n) return;
        const uint64_t k = zsort_key(P.px[p], P.py[p], P.pz[p], inv);
        const uint32_t e = P.id[p];
        klo[e]           = (uint32_t)k;
        khi[e]           = (uint32_t)(k >> 32);
        val[e]           = e;
    }
};

// AND and OR of all keys (digits on which every key agrees need no pass); acc = {and, or}, preset
// to {~0, 0}
struct k_zsort_andor {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ klo;
    const uint32_t* __restrict__ khi;
    uint32_t n;
    unsigned long long* __restrict__ acc;
    __device__ void operator()(Blk blk) const {
        __shared__ unsigned long long sa[kBlock / 64], so[kBlock / 64];
        unsigned long long a = ~0ull, o = 0ull;
        for(uint32_t i = blk.id * blockDim.x + threadIdx.x; i < n; i += blk.n * blockDim.x) {
            const unsigned long long k = (unsigned long long)khi[i] << 32 | klo[i];
            a &= k;
            o |= k;
        }
        for(int off = 32; off > 0; off >>= 1) {
            a &= __shfl_xor(a, off, 64);
            o |= __shfl_xor(o, off, 64);
        }
        if((threadIdx.x & 63) == 0) {
            sa[threadIdx.x >> 6] = a;
            so[threadIdx.x >> 6] = o;
        }
        __syncthreads();
        if(threadIdx.x == 0) {
            for(int w = 1; w < kBlock / 64; ++w) {
                a &= sa[w];
                o |= so[w];
            }
            atomicAnd(&acc[0], a);
            atomicOr(&acc[1], o);
        }
    }
};

constexpr int kRsItems = 16;                  // keys per thread per tile
constexpr int kRsTile  = kBlock * kRsItems;   // keys per tile (one workgroup)
static_assert(kBlock == 256, "the radix passes use one thread per digit value");

// digit histogram of one tile, stored digit-major: hist[d * ntiles + tile]
struct k_rs_hist {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ kw;
    uint32_t n;
    int shift;
    uint32_t ntiles;
    uint32_t* __restrict__ hist;
    __device__ void operator()(Blk blk) const {
        __shared__ uint32_t h[256];
        h[threadIdx.x] = 0;
        __syncthreads();
        const size_t base = (size_t)blk.id * kRsTile;
        for(int c = 0; c < kRsItems; ++c) {
            const size_t i = base + (size_t)c * kBlock + threadIdx.x;
            if(i < n) atomicAdd(&h[(kw[i] >> shift) & 255u], 1u);
        }
        __syncthreads();
        hist[(size_t)threadIdx.x * ntiles + blk.id] = h[threadIdx.x];
    }
};

// stable scatter of one tile: offs = exclusive scan of hist; inside the tile, keys keep their order
// (wave ballots give the rank among equal digits, earlier waves and chunks come first)
struct k_rs_scatter {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ klo;
    const uint32_t* __restrict__ khi;
    const uint32_t* __restrict__ val;
    uint32_t n;
    int word;
    int shift;
    uint32_t ntiles;
    const uint32_t* __restrict__ offs;
    uint32_t* __restrict__ olo;
    uint32_t* __restrict__ ohi;
    uint32_t* __restrict__ oval;
    __device__ void operator()(Blk blk) const {
        constexpr int       kWaves = kBlock / 64;
        __shared__ uint32_t next[256];
        __shared__ uint32_t wcnt[kWaves][256];
        const int           t = threadIdx.x, lane = t & 63, wv = t >> 6;
        next[t] = offs[(size_t)t * ntiles + blk.id];
        for(int w = 0; w < kWaves; ++w) wcnt[w][t] = 0;
        __syncthreads();
        const uint64_t below = (1ull << lane) - 1ull;
        for(int c = 0; c < kRsItems; ++c) {
            const size_t i   = (size_t)blk.id * kRsTile + (size_t)c * kBlock + t;
            const bool   act = i < n;
            uint32_t     lo = 0, hi = 0, v = 0, d = 0;
            if(act) {
                lo = klo[i];
                hi = khi[i];
                v  = val[i];
                d  = ((word ? hi : lo) >> shift) & 255u;
            }
            uint64_t peers = __ballot(act);
            for(int b = 0; b < 8; ++b) {
                const uint64_t m = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? m : ~m;
            }
            const uint32_t rank = (uint32_t)__popcll(peers & below);
            if(act && rank == 0) wcnt[wv][d] = (uint32_t)__popcll(peers);
            __syncthreads();
            if(act) {
                uint32_t pos = next[d] + rank;
                for(int w = 0; w < wv; ++w) pos += wcnt[w][d];
                olo[pos]  = lo;
                ohi[pos]  = hi;
                oval[pos] = v;
            }
            __syncthreads();
            uint32_t tot = 0;
            for(int w = 0; w < kWaves; ++w) {
                tot += wcnt[w][t];
                wcnt[w][t] = 0;
            }
            next[t] += tot;
            __syncthreads();
        }
    }
};

//==================================================================================================
// PIC_Solver::correctParticlePositions (PIC_Solver.cpp:377-485), 3-D: each particle is pushed away
// from the other particles of the 27 cells around its cell (Grid::getCellIdx, not clamped; cells
// outside the grid skipped) with w = smooth_kernel(d^2, r^2) (MathHelpers.h:661-664, (t*t)*t here),
// spring += w (p - q) / d; a pair closer than the threshold gets a random push (threshold / dt) u
// with u in [-1, 1)^3 from a hash of (seed, p, q, component), p and q being the particles' user
// indices. Then advectionSteps times pos += spring * K followed by the domain-box projection
// (BoundaryObject::constrainToBoundary(ppos), BoundaryObject.cpp:55-67). Neighbours are visited cell
// by cell (k, j, i ascending) and, in a cell, in storage order. Output to separate arrays (the
// neighbours' positions are read while others are written).
//==================================================================================================
__device__ __forceinline__ uint64_t mix64d(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ __forceinline__ float rand11(uint64_t seed, uint32_t p, uint32_t q, int comp) {
    const uint64_t h = mix64d(seed ^ mix64d(((uint64_t)p << 32 | q) * 4u + (uint64_t)comp));
    return (float)(uint32_t)(h >> 40) * (1.0f / 8388608.0f) - 1.0f;
}

struct CorrectParams {
    float    radius2, threshold, threshold2, push, K;  // push = threshold / dt
    uint32_t advSteps;
    uint64_t seed;
};

struct k_correct_positions {
    static constexpr int kThreads = kBlock;
    Particles P;
    const uint32_t* __restrict__ cell_start;
    uint32_t n;
    GridGeom g;
    BndSet bnd;
    CorrectParams c;
    float* __restrict__ ox;
    float* __restrict__ oy;
    float* __restrict__ oz;
    __device__ void operator()(Blk blk) const {
    #pragma clang fp contract(off)
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        if(p >= n) return;
        const float    x = P.px[p], y = P.py[p], z = P.pz[p];
        const uint32_t pid = P.id[p];
        const int      ci = (int)((x - g.bminx) / g.dx), cj = (int)((y - g.bminy) / g.dx), ck = (int)((z - g.bminz) / g.dx);
        float          sx = 0.f, sy = 0.f, sz = 0.f;
        for(int k = ck - 1; k <= ck + 1; ++k) {
            if(k < 0 || k >= g.nz) continue;
            for(int j = cj - 1; j <= cj + 1; ++j) {
                if(j < 0 || j >= g.ny) continue;
                for(int i = ci - 1; i <= ci + 1; ++i) {
                    if(i < 0 || i >= g.nx) continue;
                    const size_t   cell = lin3(i, j, k, g.nx, g.ny);
                    const uint32_t qb = cell_start[cell], qe = cell_start[cell + 1];
                    for(uint32_t q = qb; q < qe; ++q) {
                        if(q == p) continue;
                        const float dx = x - P.px[q], dy = y - P.py[q], dz = z - P.pz[q];
                        const float d2 = dx * dx + dy * dy + dz * dz;
                        const float x2 = d2 / c.radius2;
                        const float t  = 1.0f - x2;
                        const float w  = x2 > 1.0f ? 0.f : (t * t) * t;
                        if(d2 > c.threshold2) {
                            const float s = sqrtf(d2);
                            sx += w * dx / s;
                            sy += w * dy / s;
                            sz += w * dz / s;
                        } else {
                            const uint32_t qid = P.id[q];
                            sx += c.push * rand11(c.seed, pid, qid, 0);
                            sy += c.push * rand11(c.seed, pid, qid, 1);
                            sz += c.push * rand11(c.seed, pid, qid, 2);
                        }
                    }
                }
            }
        }
        float nx_ = x, ny_ = y, nz_ = z;
        for(uint32_t it = 0; it < c.advSteps; ++it) {
            nx_ += sx * c.K;
            ny_ += sy * c.K;
            nz_ += sz * c.K;
            float vx = 0.f, vy = 0.f, vz = 0.f;  // constrainToBoundary(ppos): no velocity
            bnd_constrain(bnd, nx_, ny_, nz_, vx, vy, vz, 0, 1.f);
        }
        ox[p] = nx_;
        oy[p] = ny_;
        oz[p] = nz_;
    }
};

// identity elements of the AND / OR key accumulators
struct k_zsort_acc_init {
    static constexpr int kThreads = 64;
    unsigned long long* __restrict__ acc;
    __device__ void operator()(Blk blk) const {
        if(threadIdx.x == 0) {
            acc[0] = ~0ull;
            acc[1] = 0ull;
        }
    }
};

// rank[perm[q]] = q, then every particle's external id becomes its rank
struct k_zsort_rank {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ perm;
    uint32_t n;
    uint32_t* __restrict__ rank;
    __device__ void operator()(Blk blk) const {
        const uint32_t q = blk.id * blockDim.x + threadIdx.x;
        if(q < n) rank[perm[q]] = q;
    }
};
struct k_zsort_rename {
    static constexpr int kThreads = kBlock;
    uint32_t* __restrict__ id;
    uint32_t n;
    const uint32_t* __restrict__ rank;
    __device__ void operator()(Blk blk) const {
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        if(p < n) id[p] = rank[id[p]];
    }
};

//--------------------------------------------------------------------------------------------------
// device-wide exclusive scan of uint32 (3 phases); tile = 256 threads x 8 items
//--------------------------------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile  = kBlock * kScanItems;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh, uint32_t& total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t  x    = v;
#pragma unroll
    for(int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if(lane >= o) x += y;
    }
    if(lane == 63) sh[wid] = x;
    __syncthreads();
    uint32_t off = 0;
    total        = 0;
    for(int w = 0; w < (int)(blockDim.x >> 6); ++w) {
        if(w < wid) off += sh[w];
        total += sh[w];
    }
    __syncthreads();
    return off + x - v;
}

struct k_scan_reduce {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ in;
    size_t n;
    uint32_t* __restrict__ partial;
    __device__ void operator()(Blk blk) const {
        __shared__ uint32_t sh[kBlock / 64];
        const size_t        base = (size_t)blk.id * kScanTile + (size_t)threadIdx.x * kScanItems;
        uint32_t            s    = 0;
    #pragma unroll
        for(int i = 0; i < kScanItems; ++i)
            if(base + i < n) s += in[base + i];
        uint32_t total;
        block_exclusive_scan(s, sh, total);
        if(threadIdx.x == 0) partial[blk.id] = total;
    }
};

// single block: exclusive scan of the per-tile partials, in chunks of 256
struct k_scan_partials {
    static constexpr int kThreads = kBlock;
    uint32_t* partial;
    uint32_t np;
    uint32_t* total_out;
    __device__ void operator()(Blk blk) const {
        __shared__ uint32_t sh[kBlock / 64];
        uint32_t            carry = 0;
        for(uint32_t b = 0; b < np; b += kBlock) {
            const uint32_t i = b + threadIdx.x;
            const uint32_t v = i < np ? partial[i] : 0u;
            uint32_t       tot;
            const uint32_t ex = block_exclusive_scan(v, sh, tot);
            if(i < np) partial[i] = carry + ex;
            carry += tot;
        }
        if(threadIdx.x == 0 && total_out) *total_out = carry;
    }
};

struct k_scan_down {
    static constexpr int kThreads = kBlock;
    const uint32_t* __restrict__ in;
    size_t n;
    const uint32_t* __restrict__ partial;
    uint32_t* __restrict__ out;
    __device__ void operator()(Blk blk) const {
        __shared__ uint32_t sh[kBlock / 64];
        const size_t        base = (size_t)blk.id * kScanTile + (size_t)threadIdx.x * kScanItems;
        uint32_t            v[kScanItems];
        uint32_t            s = 0;
    #pragma unroll
        for(int i = 0; i < kScanItems; ++i) {
            v[i] = base + i < n ? in[base + i] : 0u;
            s += v[i];
        }
        uint32_t total;
        uint32_t run = block_exclusive_scan(s, sh, total) + partial[blk.id];
    #pragma unroll
        for(int i = 0; i < kScanItems; ++i) {
            if(base + i < n) out[base + i] = run;
            run += v[i];
        }
    }
};

// Tile (tx, ty, tz) of an ntx x nty x ntz grid of tiles for workgroup blk: blocks are dispatched
// round-robin over the 8 XCDs, so each XCD is handed a contiguous run of tiles and shares the reads
// of neighbouring tiles through its own L2.
__device__ __forceinline__ void tile_of_block(Blk blk, int ntx, int nty, int ntz, int& tx, int& ty, int& tz) {
    const uint32_t nt = (uint32_t)(ntx * nty * ntz), b = blk.id, xcd = b % 8u, q = nt / 8u, r = nt % 8u;
    const uint32_t t = xcd * q + min(xcd, r) + b / 8u;
    tx = (int)(t % (uint32_t)ntx);
    ty = (int)((t / (uint32_t)ntx) % (uint32_t)nty);
    tz = (int)(t / (uint32_t)(ntx * nty));
}

//==================================================================================================
// mapParticles2Grid over cell-sorted particles (FLIP_Solver.cpp:57-95, ArrayHelpers.cpp:50-76); with
// kAffine the velocity carried to a node has the affine term of APIC_Solver.cpp:52-91 /
// AFLIP_Solver.cpp:48-90.
//
// A thread owns one column of cells (i, j) and streams up z. A particle of cell c reaches on each axis
// the nodes c, c+1 of a node-aligned grid and c-1 .. c+1 of a half-shifted one (one of the three with
// weight 0), clamps included, so all of a column's contributions fall on 18 nodes of each face grid per
// row: 2x3x3 (u), 3x2x3 (v), 3x3x2 (w). Their momentum and weight sums live in registers, a window of
// planes that moves up with the row, and each particle costs its weights and 54 multiply-adds with no
// memory traffic beyond its own record. When a plane of nodes is complete, the workgroup's columns
// exchange their partial sums through LDS and each node's owner adds its 6 (u, v) or 9 (w) columns in
// one fixed order. A node's sum is therefore: per column in (z, then particle) order, then over the
// columns by y, then x, whatever the tile, the segment length or the batch.
//
// A workgroup is 16 x 16 columns around 14 x 14 owned ones (each node needs the columns next to it:
// 1.31 visits a particle, against 1.95 for a tile of 8^3 nodes scattered into LDS, which this
// replaces) and a segment of `seg` node planes (seg + 2 rows read). Bound by VALU issue: some 210
// instructions a particle visit, and a wavefront's row lasts as long as its fullest cell. 33M particles
// at 256^3, a settling flow: 1740 -> 880 us (690 on the initial lattice, where every cell holds 8); 26k at
// 24^3, where the scattered tile was a serial chain of 27 colour rounds in 64 wavefronts: 263 -> 33 us;
// affine, 1.27M: 1155 -> 180 us (a gather per node column).
//==================================================================================================
struct FaceOut {
    float *u, *v, *w;
    uint8_t *vu, *vv, *vw;
};

constexpr int kP2gSide = 16, kP2gOwn = kP2gSide - 2;  // columns of a workgroup per axis, and those it owns

// one axis of a particle at fraction f of cell c: n = node-aligned weights of the nodes c, c+1; h =
// half-shifted weights of c-1, c, c+1. With f = x - c in [0, 1) these are bary()'s fractions without its
// branches: the base of x - 0.5 is c-1 with fraction f + 0.5 when f < 0.5, else c with f - 0.5 (both exact),
// and 1 - fraction rounds the same exact value either way.
__device__ __forceinline__ void p2g_axis(float f, float* n, float* h) {
#pragma clang fp contract(off)
    n[0] = 1.0f - f;
    n[1] = f;
    h[0] = fmaxf(0.5f - f, 0.f);
    h[1] = fminf(f + 0.5f, 1.5f - f);
    h[2] = fmaxf(f - 0.5f, 0.f);
}
// the first (lo) / last (hi) cell of an axis: outside the grid f clamps to 0 / 1 as bary's does, the
// half-shifted stencil onto the cell's own node. A coordinate that is not a number is binned to the first
// cell, and its weights are not numbers either.
__device__ __forceinline__ void p2g_axis_edge(float f, bool lo, bool hi, float* n, float* h) {
    if(!lo && !hi) return;
    p2g_axis(fminf(fmaxf(f, 0.f), 1.f), n, h);
    if(lo && h[0] > 0.f) {
        h[0] = 0.f;
        h[1] = 1.f;
    }
    if(hi) {
        if(h[2] > 0.f) h[1] = 1.f;
        h[2] = 0.f;
    }
    if(f != f) n[0] = n[1] = h[1] = h[2] = f;
}
// bary()'s weight of a node on an axis of `size` nodes, and whether the node is one of the stencil's two
__device__ __forceinline__ bool stencil_weight(float x, int size, int node, float& w) {
    int   b;
    float f;
    bary(x, size, b, f);
    w = node == b ? 1.0f - f : f;
    return node == b || node == b + 1;
}

// momentum and weight of kX x kY x kZ nodes: (wx * wy) * wz as the reference forms it, added node by node
template<int kX, int kY, int kZ>
__device__ __forceinline__ void p2g_add(const float* wx, const float* wy, const float* wz, float v, float (*m)[kX * kY], float (*w)[kX * kY]) {
#pragma clang fp contract(off)
#pragma unroll
    for(int y = 0; y < kY; ++y)
#pragma unroll
        for(int x = 0; x < kX; ++x) {
            const float ab = wx[x] * wy[y];
#pragma unroll
            for(int z = 0; z < kZ; ++z) {
                const float c = ab * wz[z];
                m[z][y * kX + x] = __builtin_fmaf(c, v, m[z][y * kX + x]);
                w[z][y * kX + x] += c;
            }
        }
}
// the same with the node's velocity v + dot(C, node - particle), the dot product in glm's order
// (APIC_Solver.cpp:73-76); dx, dy, dz: node - particle per axis
template<int kX, int kY, int kZ>
__device__ __forceinline__ void p2g_add_affine(const float* wx, const float* wy, const float* wz, float v, const float* c, const float* dx,
                                               const float* dy, const float* dz, float (*m)[kX * kY], float (*w)[kX * kY]) {
#pragma clang fp contract(off)
    float ez[kZ];
#pragma unroll
    for(int z = 0; z < kZ; ++z) ez[z] = c[2] * dz[z];
#pragma unroll
    for(int y = 0; y < kY; ++y)
#pragma unroll
        for(int x = 0; x < kX; ++x) {
            const float ab = wx[x] * wy[y], exy = c[0] * dx[x] + c[1] * dy[y];
#pragma unroll
            for(int z = 0; z < kZ; ++z) {
                const float q = ab * wz[z];
                m[z][y * kX + x] = __builtin_fmaf(q, v + (exy + ez[z]), m[z][y * kX + x]);
                w[z][y * kX + x] += q;
            }
        }
}

template<bool kAffine>
struct k_p2g {
    static constexpr int kThreads = kP2gSide * kP2gSide;
    // FLIP: 3 waves per SIMD hide a batch's load (170 registers; a batch of 4 loaded ahead of its use took
    // 206, 2 waves, and 980 us against 890 at 256^3). Affine: a record is 18 floats, so 2 waves and the next
    // record loaded ahead (bounded to 3 waves it spills: 657 against 181 us for 1.27M particles).
    static constexpr int  kOneBlocks = kAffine ? 2 : 3, kManyBlocks = kOneBlocks;
    static constexpr int  kBatch = kAffine ? 1 : 2;  // particles whose records are loaded together
    static constexpr bool kAhead = kAffine;          // ... before the batch ahead of them is added
    Particles P;
    Affine A;
    const uint32_t* __restrict__ cell_start;
    GridGeom g;
    FaceOut out;
    const uint8_t* __restrict__ occ;  // particle occupancy of the 8^3 cell bricks (binning)
    int seg;                          // node planes per workgroup
    struct Rec {
        float x[kBatch], y[kBatch], z[kBatch], u[kBatch], v[kBatch], w[kBatch];
        float p[kAffine ? kBatch : 1][3], c[kAffine ? kBatch : 1][9];
    };
    // particles [p, p + kBatch) of a cell that ends at e (a slot past it repeats the last)
    __device__ __forceinline__ void load(uint32_t p, uint32_t e, Rec& R) const {
#pragma unroll
        for(int q = 0; q < kBatch; ++q) {
            const uint32_t at = min(p + (uint32_t)q, e - 1u);
            const float4   a = P.gp[at];
            const float2   b = P.gv[at];
            R.x[q] = a.x;
            R.y[q] = a.y;
            R.z[q] = a.z;
            R.u[q] = a.w;
            R.v[q] = b.x;
            R.w[q] = b.y;
            if constexpr(kAffine) {
                R.p[q][0] = P.px[at];
                R.p[q][1] = P.py[at];
                R.p[q][2] = P.pz[at];
#pragma unroll
                for(int k = 0; k < 9; ++k) R.c[q][k] = A.c[k][at];
            }
        }
    }
    __device__ void operator()(Blk blk) const {
#pragma clang fp contract(off)
        __shared__ float2 part[21][kThreads];  // a complete plane's partial sums: u 2x3, v 3x2, w 3x3
        const int ntx = (g.nx + kP2gOwn) / kP2gOwn, nty = (g.ny + kP2gOwn) / kP2gOwn, ntz = (g.nz + seg) / seg;
        int       tx, ty, tz;
        tile_of_block(blk, ntx, nty, ntz, tx, ty, tz);
        const int  t = threadIdx.x, lx = t % kP2gSide, ly = t / kP2gSide;
        const int  i = tx * kP2gOwn - 1 + lx, j = ty * kP2gOwn - 1 + ly;  // the thread's column, and the node it owns
        const int  k0 = tz * seg, k1 = min(k0 + seg, g.nz + 1);           // node planes [k0, k1)
        const bool column = i >= 0 && i < g.nx && j >= 0 && j < g.ny;
        const bool own = lx >= 1 && lx <= kP2gOwn && ly >= 1 && ly <= kP2gOwn;
        const bool ownU = own && i <= g.nx && j < g.ny, ownV = own && i < g.nx && j <= g.ny, ownW = own && i < g.nx && j < g.ny;
        // any particle in the bricks of the cells read? One brick a thread
        const int bx0 = max(tx * kP2gOwn - 1, 0) >> 3, bx1 = min(tx * kP2gOwn + kP2gOwn, g.nx - 1) >> 3;
        const int by0 = max(ty * kP2gOwn - 1, 0) >> 3, by1 = min(ty * kP2gOwn + kP2gOwn, g.ny - 1) >> 3;
        const int bz0 = max(k0 - 1, 0) >> 3, bz1 = min(k1, g.nz - 1) >> 3;
        const int mx = bx1 - bx0 + 1, my = by1 - by0 + 1, mb = mx * my * (bz1 - bz0 + 1);
        int       any = 0;
        for(int b = t; b < mb; b += kThreads) any |= occ[((bz0 + b / (mx * my)) * g.nby + by0 + (b / mx) % my) * g.nbx + bx0 + b % mx];
        if(!__syncthreads_or(any)) {
            for(int k = k0; k < k1; ++k) {
                emit(out.u, out.vu, make_float2(0.f, 0.f), ownU && k < g.nz, lin3(i, j, k, g.nx + 1, g.ny));
                emit(out.v, out.vv, make_float2(0.f, 0.f), ownV && k < g.nz, lin3(i, j, k, g.nx, g.ny + 1));
                emit(out.w, out.vw, make_float2(0.f, 0.f), ownW, lin3(i, j, k, g.nx, g.ny));
            }
            return;
        }
        const float fi = (float)i, fj = (float)j;
        const bool  edgeXY = i == 0 || i == g.nx - 1 || j == 0 || j == g.ny - 1;
        // world positions of the column's nodes (getWorldCoordinate: (index + extra) * dx + bMin)
        float nodeX[2], halfX[3], nodeY[2], halfY[3];
        if constexpr(kAffine) {
#pragma unroll
            for(int e = 0; e < 2; ++e) {
                nodeX[e] = (fi + (float)e) * g.dx + g.bminx;
                nodeY[e] = (fj + (float)e) * g.dx + g.bminy;
            }
#pragma unroll
            for(int e = 0; e < 3; ++e) {
                halfX[e] = ((fi + (float)(e - 1)) + 0.5f) * g.dx + g.bminx;
                halfY[e] = ((fj + (float)(e - 1)) + 0.5f) * g.dx + g.bminy;
            }
        }
        // sums of the planes z-1, z, z+1 (u, v) and z, z+1 (w) while row z is read
        float mu[3][6] = {}, wu[3][6] = {}, mv[3][6] = {}, wv[3][6] = {}, mw[2][9] = {}, ww[2][9] = {};
        auto  range = [&](int z, uint32_t& b, uint32_t& e) {
            b = e = 0;
            if(column && z < g.nz) {
                const size_t c = lin3(i, j, z, g.nx, g.ny);
                b              = cell_start[c];
                e              = cell_start[c + 1];
            }
        };
        auto add = [&](const Rec& R, uint32_t p, uint32_t e, int z) {
#pragma unroll
            for(int q = 0; q < kBatch; ++q) {
                if(p + (uint32_t)q >= e) break;
                float xn[2], xh[3], yn[2], yh[3], zn[2], zh[3];
                const float fx = R.x[q] - fi, fy = R.y[q] - fj, fz = R.z[q] - (float)z;
                p2g_axis(fx, xn, xh);
                p2g_axis(fy, yn, yh);
                if(edgeXY) {
                    p2g_axis_edge(fx, i == 0, i == g.nx - 1, xn, xh);
                    p2g_axis_edge(fy, j == 0, j == g.ny - 1, yn, yh);
                }
                p2g_axis(fz, zn, zh);
                if(z == 0 || z == g.nz - 1) p2g_axis_edge(fz, z == 0, z == g.nz - 1, zn, zh);
                if constexpr(kAffine) {
                    const float fz = (float)z;
                    float       dnx[2], dhx[3], dny[2], dhy[3], dnz[2], dhz[3];
#pragma unroll
                    for(int k = 0; k < 2; ++k) {
                        dnx[k] = nodeX[k] - R.p[q][0];
                        dny[k] = nodeY[k] - R.p[q][1];
                        dnz[k] = ((fz + (float)k) * g.dx + g.bminz) - R.p[q][2];
                    }
#pragma unroll
                    for(int k = 0; k < 3; ++k) {
                        dhx[k] = halfX[k] - R.p[q][0];
                        dhy[k] = halfY[k] - R.p[q][1];
                        dhz[k] = (((fz + (float)(k - 1)) + 0.5f) * g.dx + g.bminz) - R.p[q][2];
                    }
                    p2g_add_affine<2, 3, 3>(xn, yh, zh, R.u[q], R.c[q], dnx, dhy, dhz, mu, wu);
                    p2g_add_affine<3, 2, 3>(xh, yn, zh, R.v[q], R.c[q] + 3, dhx, dny, dhz, mv, wv);
                    p2g_add_affine<3, 3, 2>(xh, yh, zn, R.w[q], R.c[q] + 6, dhx, dhy, dnz, mw, ww);
                } else {
                    p2g_add<2, 3, 3>(xn, yh, zh, R.u[q], mu, wu);
                    p2g_add<3, 2, 3>(xh, yn, zh, R.v[q], mv, wv);
                    p2g_add<3, 3, 2>(xh, yh, zn, R.w[q], mw, ww);
                }
            }
        };
        // the owned node of the planes that row k0 completes (u, v: k0 - 1; w: k0)
        const uint32_t sU = (uint32_t)((g.nx + 1) * g.ny), sV = (uint32_t)(g.nx * (g.ny + 1)), sW = (uint32_t)(g.nx * g.ny);
        uint32_t       atU = (uint32_t)(k0 - 1) * sU + (uint32_t)(j * (g.nx + 1) + i), atV = (uint32_t)(k0 - 1) * sV + (uint32_t)(j * g.nx + i),
                 atW = (uint32_t)k0 * sW + (uint32_t)(j * g.nx + i);
        float     lost = 0.f;                               // not 0 when a momentum of the owned nodes is not finite
        const int zs = max(k0 - 1, 0), ze = min(k1, g.nz);  // row nz holds no cells: it only completes the last planes
        uint32_t  pb, pe, nb, ne;
        Rec       cur, nxt;
        range(zs, pb, pe);
        if(pb < pe) load(pb, pe, cur);
        for(int z = zs; z <= ze; ++z) {
            range(z + 1, nb, ne);
            if(z == ze) ne = nb;
            // after a batch comes the cell's next one, or the first of the next row's cell
            if(pb < pe) {
                do {
                    Rec& at = kAhead ? nxt : cur;
                    if(!kAhead) add(cur, pb, pe, z);
                    if(pb + kBatch < pe) load(pb + kBatch, pe, at);
                    else if(nb < ne) load(nb, ne, at);
                    if(kAhead) {
                        add(cur, pb, pe, z);
                        cur = nxt;
                    }
                    pb += kBatch;
                } while(pb < pe);
            } else if(nb < ne) {
                load(nb, ne, cur);
            }
            pb = nb;
            pe = ne;
            // planes z-1 of u and v and z of w are complete
            if(z >= k0) {
#pragma unroll
                for(int e = 0; e < 6; ++e) {
                    part[e][t]     = make_float2(mu[0][e], wu[0][e]);
                    part[6 + e][t] = make_float2(mv[0][e], wv[0][e]);
                }
#pragma unroll
                for(int e = 0; e < 9; ++e) part[12 + e][t] = make_float2(mw[0][e], ww[0][e]);
                __syncthreads();
                if(own) {
                    // the column at (dx, dy) reaches this node with its own offset (-dx, -dy)
                    if(z > k0) {
                        float2 a = make_float2(0.f, 0.f), b = make_float2(0.f, 0.f);
#pragma unroll
                        for(int dy = -1; dy <= 1; ++dy)
#pragma unroll
                            for(int dx = -1; dx <= 0; ++dx) {
                                const float2 s = part[(1 - dy) * 2 - dx][t + dy * kP2gSide + dx];
                                a.x += s.x;
                                a.y += s.y;
                            }
#pragma unroll
                        for(int dy = -1; dy <= 0; ++dy)
#pragma unroll
                            for(int dx = -1; dx <= 1; ++dx) {
                                const float2 s = part[6 + (-dy) * 3 + 1 - dx][t + dy * kP2gSide + dx];
                                b.x += s.x;
                                b.y += s.y;
                            }
                        emit(out.u, out.vu, a, ownU, atU);
                        emit(out.v, out.vv, b, ownV, atV);
                        lost = __builtin_fmaf(b.x, 0.f, __builtin_fmaf(a.x, 0.f, lost));
                    }
                    if(z < k1) {
                        float2 c = make_float2(0.f, 0.f);
#pragma unroll
                        for(int dy = -1; dy <= 1; ++dy)
#pragma unroll
                            for(int dx = -1; dx <= 1; ++dx) {
                                const float2 s = part[12 + (1 - dy) * 3 + 1 - dx][t + dy * kP2gSide + dx];
                                c.x += s.x;
                                c.y += s.y;
                            }
                        emit(out.w, out.vw, c, ownW, atW);
                        lost = __builtin_fmaf(c.x, 0.f, lost);
                    }
                }
                __syncthreads();
                atU += sU;
                atV += sV;
                atW += sW;
            }
#pragma unroll
            for(int e = 0; e < 6; ++e) {
                mu[0][e] = mu[1][e], wu[0][e] = wu[1][e], mu[1][e] = mu[2][e], wu[1][e] = wu[2][e], mu[2][e] = 0.f, wu[2][e] = 0.f;
                mv[0][e] = mv[1][e], wv[0][e] = wv[1][e], mv[1][e] = mv[2][e], wv[1][e] = wv[2][e], mv[2][e] = 0.f, wv[2][e] = 0.f;
            }
#pragma unroll
            for(int e = 0; e < 9; ++e) mw[0][e] = mw[1][e], ww[0][e] = ww[1][e], mw[1][e] = 0.f, ww[1][e] = 0.f;
        }
        if(lost == 0.f) return;
        int at = t;
        asm volatile("" : "+v"(at));  // what follows takes no register from the loops before it
        const int ni = tx * kP2gOwn - 1 + at % kP2gSide, nj = ty * kP2gOwn - 1 + at / kP2gSide;
        for(int k = k0; k < k1; ++k)
            for(int d = 0; d < 3; ++d) {
                const int sx = g.nx + (d == 0), sy = g.ny + (d == 1), sz = g.nz + (d == 2);
                if(ni >= sx || nj >= sy || k >= sz) continue;
                float*   vel = d == 0 ? out.u : (d == 1 ? out.v : out.w);
                uint8_t* ok  = d == 0 ? out.vu : (d == 1 ? out.vv : out.vw);
                emit(vel, ok, node(d, ni, nj, k), true, lin3(ni, nj, k, sx, sy));
            }
    }
    // node velocity = momentum / weight where the weight is positive, else 0 and invalid
    __device__ __forceinline__ static void emit(float* __restrict__ vel, uint8_t* __restrict__ valid, float2 s, bool mine, size_t at) {
        if(!mine) return;
        const bool ok = s.y > kFltMin;
        vel[at]       = ok ? s.x / s.y : 0.f;
        valid[at]     = ok ? 1 : 0;
    }
    // The sums of node (i, j, k) of component d over the particles whose stencil holds it. The splat takes all
    // three nodes of a half-shifted axis and counts on a weight of 0 to add nothing, which a velocity or an
    // affine matrix that is not finite does not: the nodes of a thread that one reached (0 times their momentum
    // is not 0: three multiply-adds a plane tell) are summed again here, in the splat's order, so that it
    // reaches the eight of its stencil and the finite terms give the same bits.
    __device__ __forceinline__ float2 node(int d, int i, int j, int k) const {
#pragma clang fp contract(off)
        const float hx = d == 0 ? 0.f : 0.5f, hy = d == 1 ? 0.f : 0.5f, hz = d == 2 ? 0.f : 0.5f;
        const int   x1 = min(d == 0 ? i : i + 1, g.nx - 1), y1 = min(d == 1 ? j : j + 1, g.ny - 1), z1 = min(d == 2 ? k : k + 1, g.nz - 1);
        float2      s = make_float2(0.f, 0.f);
        for(int y = max(j - 1, 0); y <= y1; ++y)
            for(int x = max(i - 1, 0); x <= x1; ++x) {
                float2 c = make_float2(0.f, 0.f);
                for(int z = max(k - 1, 0); z <= z1; ++z) {
                    const size_t cell = lin3(x, y, z, g.nx, g.ny);
                    for(uint32_t p = cell_start[cell], e = cell_start[cell + 1]; p < e; ++p) {
                        const float4 a = P.gp[p];
                        const float2 b = P.gv[p];
                        float        wx, wy, wz;
                        const bool   in = stencil_weight(a.x - hx, g.nx + (d == 0), i, wx) & stencil_weight(a.y - hy, g.ny + (d == 1), j, wy) &
                                        stencil_weight(a.z - hz, g.nz + (d == 2), k, wz);
                        if(!in) continue;
                        float v = d == 0 ? a.w : (d == 1 ? b.x : b.y);
                        if constexpr(kAffine) {
                            const float dx = (((float)i + hx) * g.dx + g.bminx) - P.px[p], dy = (((float)j + hy) * g.dx + g.bminy) - P.py[p],
                                        dz = (((float)k + hz) * g.dx + g.bminz) - P.pz[p];
                            v = v + ((A.c[3 * d][p] * dx + A.c[3 * d + 1][p] * dy) + A.c[3 * d + 2][p] * dz);
                        }
                        const float w = (wx * wy) * wz;
                        if(w != w) return make_float2(0.f, w);  // no weight, whatever else comes
                        c.x = __builtin_fmaf(w, v, c.x);
                        c.y += w;
                    }
                }
                s.x += c.x;
                s.y += c.y;
            }
        return s;
    }
};

//==================================================================================================
// extrapolateVelocity of one component (PIC_Solver.cpp:985-1090): 4 Jacobi layers. Layer l fills an
// invalid face that is not on the array's outer layer with the mean of its neighbours valid before
// the layer (order +x, -x, +y, -y, +z, -z) and makes it valid and extrapolated.
//
// One workgroup per 8^3 brick of faces, the three components' bricks in one launch. A face changes only
// through faces within 4 face steps, so the brick and a halo of 4 faces on every side (a 16^3 tile) are
// read into LDS once and the four layers run there; they equal the two-buffer Jacobi's bit for bit. A
// halo face at distance d from the brick can go wrong (its own neighbours beyond the tile are missing)
// only from layer 4 - d on, too late to reach the brick. Faces on the tile's outer shell are never
// computed.
//
// Validity is held as one 16-bit mask per (x, y) column of the tile (bit z), in LDS for the neighbour
// columns: the faces a layer fills in a column are the invalid ones next to a set bit, a handful of bit
// operations for all 16. Those few faces go to a list that the whole workgroup then shares (they lie on
// a surface: without the list 14 threads had 14 each). Each thread reads the flags of 4 x 1 x 4 faces
// (four 4-byte loads; the columns' masks are put together in LDS) and writes back those of the same
// faces. Bound by latency: a surface brick's dependent steps (15 us at 24^3, where all run at once) and
// the flags' load of the idle ones. Both extrapolations of a substep, against one launch a component that
// tested its neighbours face by face: 116 -> 31 us at 24^3, 124 -> 41 at 64^3, 891 -> 532 at 256^3, 48
// scenes 1303 -> 654.
//
// Other workgroups read this brick's faces as their halo while it runs, so what they read as valid
// on entry is never changed: a face filled here gets its value, ext = 1 and val = gen (2 or 3, the
// host alternates it per call), which this launch's loaders read as invalid; the other generation,
// left by the previous call, reads as valid and is rewritten as 1. Every other face of the brick gets
// ext = 0. Any nonzero val therefore means valid; val holds 0 .. 3.
//==================================================================================================
typedef uint32_t uint32u __attribute__((aligned(1)));  // 4 neighbouring flags, at any address

struct ExtrapComp {
    float*   a;
    uint8_t *val, *ext;
    int      sx, sy, sz;
    uint32_t first;  // its first block, a multiple of 8; its bricks follow
    uint32_t bricks() const { return (uint32_t)(((sx + 7) / 8) * ((sy + 7) / 8) * ((sz + 7) / 8)); }
};

struct k_extrap_tile {
    static constexpr int kThreads = 256;
    static constexpr int kList = 1024;  // a longer list (scattered faces) is not made; 20 KB of LDS, 8 workgroups a CU
    static constexpr int kOneBlocks = 8, kManyBlocks = 7;  // 64 and 72 registers: 287 -> 266 us at 256^3, 48 scenes 372 -> 327
    ExtrapComp comp[3];
    uint8_t    gen;
    __device__ void operator()(Blk blk) const {
        __shared__ float    as[4096];       // 16^3, x fastest
        __shared__ union {
            uint32_t nib[4][16][4];     // [z / 4][y][x / 4]: a byte per x, a bit per z
            uint16_t list[kList];       // a layer's faces
        } u;
        __shared__ uint16_t col[256];   // the columns' valid masks
        __shared__ uint16_t fil[256];   // ... and the faces filled
        __shared__ uint32_t count[4];   // faces on the list, per layer
        const int         ci = blk.id >= comp[2].first ? 2 : (blk.id >= comp[1].first ? 1 : 0);
        const ExtrapComp& C  = comp[ci];
        const int   sx = C.sx, sy = C.sy, sz = C.sz, nbx = (sx + 7) / 8, nby = (sy + 7) / 8, nbz = (sz + 7) / 8;
        const uint32_t id = blk.id - C.first, nbk = (uint32_t)(nbx * nby * nbz);
        if(id >= nbk) return;
        int bx, by, bz;
        tile_of_block(Blk{id, nbk}, nbx, nby, nbz, bx, by, bz);
        const int      t = threadIdx.x, gi0 = bx * 8 - 4, gj0 = by * 8 - 4, gk0 = bz * 8 - 4;
        const uint32_t sxy = (uint32_t)sx * (uint32_t)sy, g4 = gen * 0x01010101u;
        // flags: faces (4 q4 .. 4 q4 + 3, fy, 4 z4 .. 4 z4 + 3) of the tile
        const int q4 = t & 3, fy = (t >> 2) & 15, z4 = t >> 6, fi = gi0 + 4 * q4, fj = gj0 + fy;
        const bool rowIn = fj >= 0 && fj < sy, whole = fi >= 0 && fi + 4 <= sx;
        auto       at = [&](int q) { return (uint32_t)(gk0 + 4 * z4 + q) * sxy + (uint32_t)fj * (uint32_t)sx + (uint32_t)fi; };
        auto       zIn = [&](int q) { return rowIn && (uint32_t)(gk0 + 4 * z4 + q) < (uint32_t)sz; };
        uint32_t   v0[4], ok[4], acc = 0;  // flags on entry; 1 per valid face, per byte
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            v0[q] = 0;
            if(!zIn(q)) continue;
            if(whole) v0[q] = *reinterpret_cast<const uint32u*>(C.val + at(q));
            else
                for(int e = 0; e < 4; ++e)
                    if((uint32_t)(fi + e) < (uint32_t)sx) v0[q] |= (uint32_t)C.val[at(q) + e] << (8 * e);
        }
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            const uint32_t x = v0[q] ^ g4;
            ok[q]            = (v0[q] | v0[q] >> 1) & (x | x >> 1) & 0x01010101u;  // neither 0 nor gen
            acc |= ok[q] << q;
        }
        u.nib[z4][fy][q4] = acc;
        if(t < 4) count[t] = 0;
        bool work = __syncthreads_or(acc != 0) != 0;
        // the thread's column of the tile
        const int x = t & 15, y = t >> 4, gi = gi0 + x, gj = gj0 + y;
        uint32_t  m = 0;  // valid faces
        if(work) {
#pragma unroll
            for(int k = 0; k < 4; ++k) m |= (u.nib[k][y][x >> 2] >> (8 * (x & 3)) & 15u) << (4 * k);
            col[t] = (uint16_t)m;
            const uint32_t inZ = (gk0 < 0 ? 0xFFF0u : 0xFFFFu) & (sz - gk0 < 16 ? (1u << (sz - gk0)) - 1u : 0xFFFFu);
            const bool     open = x >= 4 && x < 12 && y >= 4 && y < 12 && gi < sx && gj < sy && (~m & inZ & 0x0FF0u) != 0;
            work                = __syncthreads_or(open) != 0;
        }
        if(work) {
            // faces that can be filled: not on the tile's outer shell, not on the array's outer layer
            const int zl = max(1, 1 - gk0), zh = min(14, sz - 2 - gk0);
            uint32_t  can = zl <= zh ? ((2u << zh) - 1u) & ~((1u << zl) - 1u) & ~m : 0u;
            if(x < 1 || x > 14 || y < 1 || y > 14 || gi < 1 || gi > sx - 2 || gj < 1 || gj > sy - 2) can = 0;
            // the values of the faces valid on entry (the others are written before they are read)
            const uint32_t c0 = (uint32_t)gj * (uint32_t)sx + (uint32_t)gi;
#pragma unroll
            for(int z = 0; z < 16; ++z)
                if(m >> z & 1u) as[(z << 8) | t] = C.a[(uint32_t)(gk0 + z) * sxy + c0];
            uint32_t filled = 0;
            // Layer l (0 .. 3) fills only the faces within 3 - l cells (per axis) of the brick: a face
            // farther out reaches the brick through fewer than the layers left, so leaving it unfilled
            // changes no brick face, and every face a layer reads lies within the previous layer's region.
            for(int layer = 0; layer < 4; ++layer) {
                const int lo = layer + 1, hi = 14 - layer;
                uint32_t  fill = 0;
                if(x >= lo && x <= hi && y >= lo && y <= hi)
                    fill = ((uint32_t)col[t + 1] | col[t - 1] | col[t + 16] | col[t - 16] | m >> 1 | m << 1) & can & ((2u << hi) - 1u) & ~((1u << lo) - 1u);
                // list positions: the lanes before this one in the wavefront, one LDS atomic a wavefront
                uint32_t n = __popc(fill), pre = n;
#pragma unroll
                for(int o = 1; o < 64; o <<= 1) {
                    const uint32_t up = __shfl_up(pre, o, 64);
                    if((t & 63) >= o) pre += up;
                }
                uint32_t base = 0;
                if((t & 63) == 63 && pre) base = atomicAdd(&count[layer], pre);
                uint32_t pos = __shfl(base, 63, 64) + pre - n;
                for(uint32_t f = fill; f && pos < (uint32_t)kList; f &= f - 1u) u.list[pos++] = (uint16_t)(__builtin_ctz(f) << 8 | t);
                __syncthreads();
                auto face = [&](int q) {
                    const int      z = q >> 8, c = q & 255;
                    // neighbours in the order +x, -x, +y, -y, +z, -z, those valid before the layer
                    const uint32_t own = col[c];
                    const uint32_t k[6] = {(uint32_t)col[c + 1] >> z & 1u, (uint32_t)col[c - 1] >> z & 1u, (uint32_t)col[c + 16] >> z & 1u,
                                           (uint32_t)col[c - 16] >> z & 1u, own >> (z + 1) & 1u, own >> (z - 1) & 1u};
                    const float    v[6] = {as[q + 1], as[q - 1], as[q + 16], as[q - 16], as[q + 256], as[q - 256]};
                    float          sum = 0.f;  // starts at +0 and never becomes -0, so adding +0 for a neighbour not taken is exact
                    uint32_t       num = 0;
#pragma unroll
                    for(int d = 0; d < 6; ++d) {
                        sum += k[d] ? v[d] : 0.f;
                        num += k[d];
                    }
                    as[q] = sum / (float)num;  // a face filled by a layer is not read by it
                };
                const uint32_t total = count[layer];
                if(total <= (uint32_t)kList)
                    for(uint32_t e = t; e < total; e += kThreads) face(u.list[e]);
                else
                    for(uint32_t f = fill; f; f &= f - 1u) face(__builtin_ctz(f) << 8 | t);
                __syncthreads();
                m |= fill;
                can &= ~fill;
                filled |= fill;
                col[t] = (uint16_t)m;
                if(total == 0) break;  // nothing left within reach
                __syncthreads();
            }
            fil[t] = (uint16_t)filled;
            if(x >= 4 && x < 12 && y >= 4 && y < 12)
                for(uint32_t f = filled & 0x0FF0u; f; f &= f - 1u) {
                    const int z = __builtin_ctz(f);
                    C.a[(uint32_t)(gk0 + z) * sxy + c0] = as[(z << 8) | t];
                }
            __syncthreads();
        }
        // flags of the brick's faces
        if(q4 < 1 || q4 > 2 || fy < 4 || fy >= 12 || z4 < 1 || z4 > 2) return;
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            if(!zIn(q)) continue;
            uint32_t f = 0;
            if(work)
#pragma unroll
                for(int e = 0; e < 4; ++e) f |= ((uint32_t)fil[fy * 16 + 4 * q4 + e] >> (4 * z4 + q) & 1u) << (8 * e);
            const uint32_t set = (ok[q] | f) * 255u, nv = (v0[q] & ~set) | ok[q] | f * gen;
            if(whole) {
                *reinterpret_cast<uint32u*>(C.ext + at(q)) = f;
                if(nv != v0[q]) *reinterpret_cast<uint32u*>(C.val + at(q)) = nv;
            } else {
                for(int e = 0; e < 4; ++e)
                    if((uint32_t)(fi + e) < (uint32_t)sx) {
                        C.ext[at(q) + e] = (uint8_t)(f >> (8 * e));
                        if((nv ^ v0[q]) >> (8 * e) & 255u) C.val[at(q) + e] = (uint8_t)(nv >> (8 * e));
                    }
            }
        }
    }
};

//==================================================================================================
// constrainGridVelocity, component d (PIC_Solver.cpp:1094-1115, ArrayHelpers.cpp:214-251)
//==================================================================================================
__device__ __forceinline__ void interp_gradient(const float* __restrict__ b, int sx, int sy, int sz, float x, float y, float z,
                                                float& gx, float& gy, float& gz) {
    int   i, j, k;
    float fi, fj, fk;
    bary(x, sx, i, fi);
    bary(y, sy, j, fj);
    bary(z, sz, k, fk);
    auto  at   = [&](int a, int c, int e) { return b[lin3(a, c, e, sx, sy)]; };
    float v000 = at(i, j, k), v001 = at(i, j, k + 1), v010 = at(i, j + 1, k), v011 = at(i, j + 1, k + 1);
    float v100 = at(i + 1, j, k), v101 = at(i + 1, j, k + 1), v110 = at(i + 1, j + 1, k), v111 = at(i + 1, j + 1, k + 1);
    gx = bilerpf(v100 - v000, v110 - v010, v101 - v001, v111 - v011, fj, fk);
    gy = bilerpf(v010 - v000, v110 - v100, v011 - v001, v111 - v101, fi, fk);
    gz = bilerpf(v001 - v000, v101 - v100, v011 - v010, v111 - v110, fi, fj);
}

// A face is constrained where the extrapolation filled it and its weight is 0. The new value of such a face
// goes to tmp first: the interpolation around one face reads its neighbours, which must hold the values
// from before this component's pass, but those of the components passed before it (components u, v, w in
// turn): they are taken from their tmp. One pass over the faces applies all three afterwards (k_faces).
struct FaceComp {
    float*         vel;
    float*         tmp;
    const uint8_t* ext;
    const float*   weight;
};
__device__ __forceinline__ bool constrained(uint8_t ext, float weight) { return ext == 1 && weight < kFltMin; }

// the stencil's corners of a component whose new values may still lie in tmp
__device__ __forceinline__ Corners corners_constrained(const FaceComp& c, const Stencil& s) {
    Corners r = corners(c.vel, s);
    const Corners t = corners(c.tmp, s), w = corners(c.weight, s);
    const size_t  at[8] = {s.at, s.at + 1, s.at + s.sx, s.at + s.sx + 1, s.at + s.sxy, s.at + s.sxy + 1, s.at + s.sxy + s.sx, s.at + s.sxy + s.sx + 1};
#pragma unroll
    for(int e = 0; e < 8; ++e) r.v[e] = constrained(c.ext[at[e]], w.v[e]) ? t.v[e] : r.v[e];
    return r;
}

// The few faces to constrain (about one in a thousand) are listed by the workgroup's first look at the flags
// and weights of its 1024 faces and then shared by its threads, one each: four in turn in the thread that
// found them took 11 us a component at 24^3, this takes 7.
struct k_constrain {
    static constexpr int kThreads = kBlock;
    FaceComp c[3];
    GridGeom g;
    int d;
    const float* __restrict__ bsdf;
    // the new velocity of face t
    __device__ __forceinline__ float face(uint32_t t, int sx, int sy) const {
        float val = c[d].vel[t];
        int i, j, k;
        unlin3(t, sx, sy, i, j, k);
        float gp[3] = {(float)i + 0.5f, (float)j + 0.5f, (float)k + 0.5f};
        gp[d]       = d == 0 ? (float)i : (d == 1 ? (float)j : (float)k);
        const Stencil su = stencil3(g.nx + 1, g.ny, g.nz, gp[0], gp[1] - 0.5f, gp[2] - 0.5f);
        const Stencil sv = stencil3(g.nx, g.ny + 1, g.nz, gp[0] - 0.5f, gp[1], gp[2] - 0.5f);
        const Stencil sw = stencil3(g.nx, g.ny, g.nz + 1, gp[0] - 0.5f, gp[1] - 0.5f, gp[2]);
        float vx = interp8(d > 0 ? corners_constrained(c[0], su) : corners(c[0].vel, su), su);
        float vy = interp8(d > 1 ? corners_constrained(c[1], sv) : corners(c[1].vel, sv), sv);
        float vz = interp8(corners(c[2].vel, sw), sw);
        float nx, ny, nz;
        interp_gradient(bsdf, g.nx + 1, g.ny + 1, g.nz + 1, gp[0], gp[1], gp[2], nx, ny, nz);
        const float m2 = nx * nx + ny * ny + nz * nz;
        if(m2 > kFltMin) {
            const float s = sqrtf(m2);
            nx /= s;
            ny /= s;
            nz /= s;
            const float dt = vx * nx + vy * ny + vz * nz;
            vx -= dt * nx;
            vy -= dt * ny;
            vz -= dt * nz;
            val = d == 0 ? vx : (d == 1 ? vy : vz);
        }
        return val;
    }
    __device__ void operator()(Blk blk) const {
        __shared__ uint16_t list[4 * kThreads];
        __shared__ uint32_t count;
        const int      sx = g.nx + (d == 0), sy = g.ny + (d == 1), sz = g.nz + (d == 2), t = threadIdx.x;
        const uint32_t N = (uint32_t)sx * (uint32_t)sy * (uint32_t)sz, b0 = blk.id * 4u * kThreads, t0 = b0 + 4u * (uint32_t)t;
        uint32_t       hit = 0;
        if(t0 + 4 <= N) {
            const uchar4 e = *reinterpret_cast<const uchar4*>(c[d].ext + t0);
            if(e.x == 1 || e.y == 1 || e.z == 1 || e.w == 1) {
                const float4 w = *reinterpret_cast<const float4*>(c[d].weight + t0);
                hit = (constrained(e.x, w.x) ? 1u : 0u) | (constrained(e.y, w.y) ? 2u : 0u) | (constrained(e.z, w.z) ? 4u : 0u) |
                      (constrained(e.w, w.w) ? 8u : 0u);
            }
        } else {
            for(uint32_t f = t0; f < N; ++f)
                if(constrained(c[d].ext[f], c[d].weight[f])) hit |= 1u << (f - t0);
        }
        if(t == 0) count = 0;
        if(!__syncthreads_or((int)hit)) return;
        if(hit) {
            uint32_t at = atomicAdd(&count, (uint32_t)__popc(hit));
            for(uint32_t h = hit; h; h &= h - 1u) list[at++] = (uint16_t)(4 * t + __builtin_ctz(h));
        }
        __syncthreads();
        for(uint32_t e = t; e < count; e += kThreads) {
            const uint32_t f = b0 + list[e];
            c[d].tmp[f]      = face(f, sx, sy);
        }
    }
};

// One pass over all faces for what a substep does to each on its own: the constrained faces take their new
// values (apply), the velocities are backed up (old, FLIP_Data.h:48-52) and a constant gravity is added
// (add[d]; PIC_Solver.cpp:505-529). Four faces a thread.
struct k_faces {
    static constexpr int kThreads = kBlock;
    FaceComp c[3];
    float*   old[3];     // null: no backup
    uint32_t n[3], first[3];  // faces, first block
    int      apply, gravity;  // gravity: bit d, add[d] to component d
    float    add[3];
    static uint32_t blocks(uint32_t n) { return (n + 4 * kThreads - 1) / (4 * kThreads); }
    __device__ void operator()(Blk blk) const {
        const int      d  = blk.id >= first[2] ? 2 : (blk.id >= first[1] ? 1 : 0);
        const uint32_t t0 = 4u * ((blk.id - first[d]) * kThreads + threadIdx.x), N = n[d];
        if(t0 >= N) return;
        const FaceComp C = c[d];
        const float    a = add[d];
        const bool     on = gravity >> d & 1;
        if(t0 + 4 <= N) {
            const bool whole = old[d] || on;
            uint32_t   hit = 0;
            if(apply) {
                const uchar4 e = *reinterpret_cast<const uchar4*>(C.ext + t0);
                if(e.x == 1 || e.y == 1 || e.z == 1 || e.w == 1) {
                    const float4 w = *reinterpret_cast<const float4*>(C.weight + t0);
                    hit = (constrained(e.x, w.x) ? 1u : 0u) | (constrained(e.y, w.y) ? 2u : 0u) | (constrained(e.z, w.z) ? 4u : 0u) |
                          (constrained(e.w, w.w) ? 8u : 0u);
                }
            }
            if(!whole && !hit) return;
            float4 v = *reinterpret_cast<const float4*>(C.vel + t0);
            if(hit & 1u) v.x = C.tmp[t0];
            if(hit & 2u) v.y = C.tmp[t0 + 1];
            if(hit & 4u) v.z = C.tmp[t0 + 2];
            if(hit & 8u) v.w = C.tmp[t0 + 3];
            if(old[d]) *reinterpret_cast<float4*>(old[d] + t0) = v;
            if(on) {
                v.x += a;
                v.y += a;
                v.z += a;
                v.w += a;
            }
            if(hit || on) *reinterpret_cast<float4*>(C.vel + t0) = v;
        } else {
            for(uint32_t t = t0; t < N; ++t) {
                float v = C.vel[t];
                if(apply && constrained(C.ext[t], C.weight[t])) v = C.tmp[t];
                if(old[d]) old[d][t] = v;
                C.vel[t] = on ? v + a : v;
            }
        }
    }
};

//==================================================================================================
// addGravity (PIC_Solver.cpp:505-529): Earth / Directional add a constant per component (k_faces)
//==================================================================================================
// c = a * b elementwise
struct k_mul_arrays {
    static constexpr int kThreads = kBlock;
    const float* __restrict__ a;
    const float* __restrict__ b;
    float* __restrict__ c;
    size_t n;
    __device__ void operator()(Blk blk) const {
        const size_t i = (size_t)blk.id * blockDim.x + threadIdx.x;
        if(i < n) c[i] = a[i] * b[i];
    }
};

// ToCenter / FromCenter: the reference walks velocities[0]'s index range for every component
// (PIC_Solver.cpp:521); indices outside component d's array are skipped here.
struct k_gravity_center {
    static constexpr int kThreads = kBlock;
    float* __restrict__ a;
    GridGeom g;
    int d;
    float cx;
    float cy;
    float cz;
    int toCenter;
    float dt;
    __device__ void operator()(Blk blk) const {
        const int    sx = g.nx + 1, sy = g.ny, sz = g.nz;
        const size_t t  = (size_t)blk.id * blockDim.x + threadIdx.x;
        if(t >= (size_t)sx * sy * sz) return;
        int i, j, k;
        unlin3((uint32_t)t, sx, sy, i, j, k);
        const int ax = g.nx + (d == 0), ay = g.ny + (d == 1), az = g.nz + (d == 2);
        if(i >= ax || j >= ay || k >= az) return;
        float gp[3] = {(float)i + 0.5f, (float)j + 0.5f, (float)k + 0.5f};
        gp[d]       = d == 0 ? (float)i : (d == 1 ? (float)j : (float)k);
        const float wx = gp[0] * g.dx + g.bminx, wy = gp[1] * g.dx + g.bminy, wz = gp[2] * g.dx + g.bminz;
        float       dv[3];
        dv[0]          = toCenter ? cx - wx : wx - cx;
        dv[1]          = toCenter ? cy - wy : wy - cy;
        dv[2]          = toCenter ? cz - wz : wz - cz;
        const float is = 1.0f / sqrtf(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2]);
        a[lin3(i, j, k, ax, ay)] += (9.81f * (dv[d] * is)) * dt;
    }
};

//==================================================================================================
// computeCellWeights (PIC_Solver.cpp:543-597); counts faces with weight < FLT_MIN (solid faces)
//==================================================================================================
struct k_weights {
    static constexpr int kThreads = kBlock;
    const float* __restrict__ b;
    GridGeom g;
    float* __restrict__ wu;
    float* __restrict__ wv;
    float* __restrict__ ww;
    uint32_t* solidFaces;
    __device__ void operator()(Blk blk) const {
        const int    sx = g.nx + 1, sy = g.ny + 1, sz = g.nz + 1;
        const size_t t  = (size_t)blk.id * blockDim.x + threadIdx.x;
        if(t >= (size_t)sx * sy * sz) return;
        int i, j, k;
        unlin3((uint32_t)t, sx, sy, i, j, k);
        auto      B = [&](int a, int c, int e) { return b[lin3(a, c, e, sx, sy)]; };
        uint32_t  solid = 0;
        if(j < g.ny && k < g.nz) {
            float w = clamp01f(1.0f - fraction_inside4(B(i, j, k), B(i, j + 1, k), B(i, j, k + 1), B(i, j + 1, k + 1)));
            wu[lin3(i, j, k, g.nx + 1, g.ny)] = w;
            solid += w < kFltMin;
        }
        if(i < g.nx && k < g.nz) {
            float w = clamp01f(1.0f - fraction_inside4(B(i, j, k), B(i, j, k + 1), B(i + 1, j, k), B(i + 1, j, k + 1)));
            wv[lin3(i, j, k, g.nx, g.ny + 1)] = w;
            solid += w < kFltMin;
        }
        if(i < g.nx && j < g.ny) {
            float w = clamp01f(1.0f - fraction_inside4(B(i, j, k), B(i, j + 1, k), B(i + 1, j, k), B(i + 1, j + 1, k)));
            ww[lin3(i, j, k, g.nx, g.ny)] = w;
            solid += w < kFltMin;
        }
        if(solid) atomicAdd(solidFaces, solid);
    }
};

// computeBoundarySDF: the smallest signed distance over the boundary objects (PIC_Solver.cpp:1158-1168)
struct k_boundary_sdf {
    static constexpr int kThreads = kBlock;
    float* __restrict__ b;
    GridGeom g;
    BndSet bnd;
    __device__ void operator()(Blk blk) const {
        const int    sx = g.nx + 1, sy = g.ny + 1, sz = g.nz + 1;
        const size_t t  = (size_t)blk.id * blockDim.x + threadIdx.x;
        if(t >= (size_t)sx * sy * sz) return;
        int i, j, k;
        unlin3((uint32_t)t, sx, sy, i, j, k);
        const float x = (float)i * g.dx + g.bminx, y = (float)j * g.dx + g.bminy, z = (float)k * g.dx + g.bminz;
        float       m = 3.40282347e+38f;  // Huge<float>
        for(int q = 0; q < bnd.nGroups; ++q) m = smin(m, bnd_group_sd(bnd, q, x, y, z));
        b[t] = m;
    }
};

//==================================================================================================
// computeFluidSDF as a gather (PIC_Solver.cpp:601-689): phi(c) = min over particles whose clamped
// 3x3x3 window holds c of |centre(c) - p| - sdfRadius; min is exact, so the result is bit-identical
// to the reference's locked scatter. Then the solid extension. A work-group owns an 8x8x4 tile of
// cells; tiles are handed out so that each XCD (blocks are dispatched round-robin over 8 XCDs) works
// on a contiguous run of tiles and shares neighbour-cell reads through its own L2. A cell visits its
// own cell first and stops as soon as no farther neighbour can lower the minimum, so most cells read
// only their own particles (staging the 10x10x6 halo in LDS cost more than it saved). Bound by the
// latency of its dependent reads (cell range, particles), so particles are read eight at a time and the
// cells that need their neighbours (at the surface) share out their nine rows over the workgroup. 33M
// particles at 256^3: 547 -> 285 us; 5.7M at 160x120x130: 135 -> 67; 26k at 24^3: 50 -> 25.
//==================================================================================================
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kTileX = 8, kTileY = 8, kTileZ = 4;
constexpr int kTileThreads = kTileX * kTileY * kTileZ;  // 256

struct k_fluid_sdf {
    static constexpr int kThreads = kTileThreads;
    Particles P;
    const uint32_t* __restrict__ cell_start;
    GridGeom g;
    const float* __restrict__ bsdf;
    float* __restrict__ phi;
    const uint8_t* __restrict__ occ;  // particle occupancy of the 8^3 cell bricks (the same binning)
    __device__ void operator()(Blk blk) const {
        const int ntx = (g.nx + kTileX - 1) / kTileX, nty = (g.ny + kTileY - 1) / kTileY, ntz = (g.nz + kTileZ - 1) / kTileZ;
        int       tx, ty, tz;
        tile_of_block(blk, ntx, nty, ntz, tx, ty, tz);
        __shared__ uint32_t bits[kTileThreads];  // the cells' smallest squares
        __shared__ uint8_t  list[kTileThreads];
        __shared__ uint32_t nList;
        const int t = threadIdx.x, x0 = tx * kTileX, y0 = ty * kTileY, z0 = tz * kTileZ;
        const int i = x0 + t % kTileX, j = y0 + (t / kTileX) % kTileY, k = z0 + t / (kTileX * kTileY);
        const bool in = i < g.nx && j < g.ny && k < g.nz;
        // Only the smallest squared distance is tracked: the square root and the subtraction of the radius
        // are monotonic as rounded, so the minimum of the distances is that of the smallest square.
        // Smallest square of the particles [b, e) from the centre of cell (i, j, k), eight at a time: 4-wide
        // loads at any particle (the arrays are padded for them).
        auto visit = [&](int i, int j, int k, uint32_t b, uint32_t e, float least) {
            const float sx = ((float)i + 0.5f) * g.dx + g.bminx;
            const float sy = ((float)j + 0.5f) * g.dx + g.bminy;
            const float sz = ((float)k + 0.5f) * g.dx + g.bminz;
            // next to the grid's edge, particles may be clamped into a boundary cell: their true window counts
            const bool edge = i <= 1 || j <= 1 || k <= 1 || i >= g.nx - 2 || j >= g.ny - 2 || k >= g.nz - 2;
            const float hix = 0.9999f * ((float)g.nx * g.dx), hiy = 0.9999f * ((float)g.ny * g.dx), hiz = 0.9999f * ((float)g.nz * g.dx);
            for(uint32_t p = b; p < e; p += 8) {
                float4u x[2], y[2], z[2];
#pragma unroll
                for(int h = 0; h < 2; ++h) {
                    const uint32_t q = h && p + 4 < e ? p + 4 : p;
                    x[h]             = *reinterpret_cast<const float4u*>(P.px + q);
                    y[h]             = *reinterpret_cast<const float4u*>(P.py + q);
                    z[h]             = *reinterpret_cast<const float4u*>(P.pz + q);
                }
#pragma unroll
                for(int h = 0; h < 2; ++h)
#pragma unroll
                    for(int q = 0; q < 4; ++q) {
                        bool counts = p + 4 * h + q < e;
                        const float ux = x[h][q] - g.bminx, uy = y[h][q] - g.bminy, uz = z[h][q] - g.bminz;
                        if(edge && (!(fminf(fminf(ux, uy), uz) >= 0.f) || !(ux < hix && uy < hiy && uz < hiz))) {  // maybe outside the grid
                            const int ci = (int)(ux / g.dx), cj = (int)(uy / g.dx), ck = (int)(uz / g.dx);
                            counts &= i >= ci - 1 && i <= ci + 1 && j >= cj - 1 && j <= cj + 1 && k >= ck - 1 && k <= ck + 1;
                        }
                        const float dx = sx - x[h][q], dy = sy - y[h][q], dz = sz - z[h][q];
                        const float d2 = dx * dx + dy * dy + dz * dz;
                        least          = counts ? fminf(least, d2) : least;
                    }
            }
            return least;
        };
        // The own cell first. Then the rows (3 cells along x) through its face neighbours, and those through
        // its edge and corner neighbours: no particle of these is nearer to the centre than 0.5 or 0.7071 dx
        // (less 1e-3 dx for the rounding of particle-to-cell assignment), so once the nearest particle found
        // beats that bound they cannot lower the minimum. min() is exact, so visiting fewer cells, in any
        // order, gives the same bits.
        const float b1 = 0.499f * g.dx, b2 = 0.7061068f * g.dx;
        float       least = 3.40282347e+38f;
        bool        more  = false;
        if(t == 0) nList = 0;
        __syncthreads();
        if(in) {
            // no particle in the bricks that hold the 3x3x3 cells around this one: nothing to visit, the
            // distance stays at its initial value (the scan below would find every cell empty)
            const int bx0 = max(i - 1, 0) >> 3, bx1 = min(i + 1, g.nx - 1) >> 3, by0 = max(j - 1, 0) >> 3, by1 = min(j + 1, g.ny - 1) >> 3;
            const int bz0 = max(k - 1, 0) >> 3, bz1 = min(k + 1, g.nz - 1) >> 3;
            uint32_t  near = 0;
#pragma unroll
            for(int e = 0; e < 8; ++e) near |= occ[((e & 4 ? bz1 : bz0) * g.nby + (e & 2 ? by1 : by0)) * g.nbx + (e & 1 ? bx1 : bx0)];
            if(near) {
                const size_t c = lin3(i, j, k, g.nx, g.ny);
                least          = visit(i, j, k, cell_start[c], cell_start[c + 1], least);
                more           = !(least < b1 * b1);
            }
        }
        // the cells that need their neighbours go to a list, and the workgroup shares their rows
        {
            const uint64_t m = __ballot(more);
            uint32_t       at = 0;
            if((t & 63) == 0 && m) at = atomicAdd(&nList, (uint32_t)__popcll(m));
            at = __shfl(at, 0, 64);
            if(more) list[at + (uint32_t)__popcll(m & ((1ull << (t & 63)) - 1ull))] = (uint8_t)t;
            bits[t] = __float_as_uint(least);
        }
        __syncthreads();
        const uint32_t n = nList;
        for(uint32_t task = t; task < 9u * n; task += kTileThreads) {
            const uint32_t r = task / n, cell = list[task - r * n];  // row r of one cell after the other
            if(r >= 5 && __uint_as_float(bits[cell]) < b2 * b2) continue;
            const int ci = x0 + (int)cell % kTileX, cj = y0 + ((int)cell / kTileX) % kTileY, ck = z0 + (int)cell / (kTileX * kTileY);
            // own row, the four through face neighbours, the four beyond
            const int y = cj + ((r == 1 || r == 5 || r == 7) ? -1 : (r == 2 || r == 6 || r == 8) ? 1 : 0);
            const int z = ck + ((r == 3 || r == 5 || r == 6) ? -1 : (r == 4 || r == 7 || r == 8) ? 1 : 0);
            if(y < 0 || y >= g.ny || z < 0 || z >= g.nz) continue;
            const size_t at = lin3(0, y, z, g.nx, g.ny);
            const float  d  = visit(ci, cj, ck, cell_start[at + max(ci - 1, 0)], cell_start[at + min(ci + 1, g.nx - 1) + 1], 3.40282347e+38f);
            atomicMin(&bits[cell], __float_as_uint(d));  // nonnegative floats order as their bits
        }
        __syncthreads();
        if(!in) return;
        least = __uint_as_float(bits[t]);
        float       best = g.dx * 3.0f;
        const float v    = sqrtf(least) - g.sdfRadius;
        if(least < 3.0e+38f && v < best) best = v;
        if(best < g.halfdx) {
            const int   sxn = g.nx + 1, syn = g.ny + 1;
            auto        B   = [&](int a, int c, int e) { return bsdf[lin3(a, c, e, sxn, syn)]; };
            const float s   = 0.125f * (B(i, j, k) + B(i + 1, j, k) + B(i, j + 1, k) + B(i + 1, j + 1, k) + B(i, j, k + 1) +
                                      B(i + 1, j, k + 1) + B(i, j + 1, k + 1) + B(i + 1, j + 1, k + 1));
            if(s < 0) best = -g.halfdx;
        }
        phi[lin3(i, j, k, g.nx, g.ny)] = best;
    }
};

//==================================================================================================
// Pressure bricks
//==================================================================================================
// Fluid cells per brick, one wavefront a brick (two 4-cell loads a lane), and the coarse levels' flags: a
// coarse brick is active when a fluid brick lies below it, and the level-l brick of (bx, by, bz) is
// (bx >> l, by >> l, bz >> l). Each writes the value 1, so concurrent writes to one flag agree.
constexpr int kMaxMgLevels = 16;
struct k_brick_flags {
    static constexpr int kThreads = kBlock;
    const float* __restrict__ phi;
    GridGeom  g;
    uint32_t* count;   // per brick
    int       nLevels; // coarse levels 1 .. nLevels, their flags cleared before
    int       cnbx[kMaxMgLevels], cnby[kMaxMgLevels];
    uint32_t* flag[kMaxMgLevels];
    static uint32_t blocks(uint32_t nb) { return (nb + kThreads / 64 - 1) / (kThreads / 64); }
    __device__ void operator()(Blk blk) const {
        const int lane = threadIdx.x & 63, b = blk.id * (kThreads / 64) + (threadIdx.x >> 6);
        if(b >= g.nbx * g.nby * g.nbz) return;
        const int bx = b % g.nbx, by = (b / g.nbx) % g.nby, bz = b / (g.nbx * g.nby);
        uint32_t  n = 0;
#pragma unroll
        for(int h = 0; h < 2; ++h) {
            const int e = lane + 64 * h, i = bx * 8 + 4 * (e & 1), j = by * 8 + ((e >> 1) & 7), k = bz * 8 + (e >> 4);
            float4u   v = {0.f, 0.f, 0.f, 0.f};
            if(j < g.ny && k < g.nz) {
                const size_t at = lin3(i, j, k, g.nx, g.ny);
                if(i + 4 <= g.nx) v = *reinterpret_cast<const float4u*>(phi + at);
                else
                    for(int q = 0; q < 4; ++q)
                        if(i + q < g.nx) v[q] = phi[at + q];
            }
#pragma unroll
            for(int q = 0; q < 4; ++q) n += (uint32_t)__popcll(__ballot(v[q] < 0.f));
        }
        if(lane != 0) return;
        count[b] = n;
        if(n)
            for(int l = 1; l <= nLevels; ++l) flag[l][((bz >> l) * cnby[l] + (by >> l)) * cnbx[l] + (bx >> l)] = 1u;
    }
};

// Slots of the active bricks of every level, one workgroup a level (with the flags and tables 3 launches and
// one host wait where a three-launch scan, slot, neighbour and parent table kernel per level and two waits
// took 150 us of a 64^3 substep's 2350, and the cell counts' one atomic 121 us at 256^3): slots in ascending brick order, the
// brick -> slot (-1: inactive) and slot -> brick tables, and the level's count to out[1 + l]. Level 0 reads
// the cell counts and adds them up to out[0]; the coarse levels' flags return to 0 for the next time. Its time
// grows with the brick grid: 41 us at 256^3, 277 at 512^3, 1490 at 900^3. With the flags and tables that is still
// less than the flags, scans and tables before it at each (427 against 544 us at 512^3, 2230 against 2520 at 900^3).
struct k_brick_index {
    static constexpr int kThreads = 1024, kItems = 8;
    uint32_t* flag[kMaxMgLevels];
    int32_t * brickSlot[kMaxMgLevels], *slotBrick[kMaxMgLevels];
    uint32_t  nb[kMaxMgLevels];
    uint32_t* out;
    __device__ void operator()(Blk blk) const {
        __shared__ uint32_t sh[kThreads / 64];
        const int           l = (int)blk.id;
        const uint32_t      n = nb[l];
        uint32_t*           f = flag[l];
        uint32_t            carry = 0, cells = 0;
        for(uint32_t b0 = 0; b0 < n; b0 += kThreads * kItems) {
            const uint32_t b = b0 + threadIdx.x * kItems;
            uint32_t       v[kItems], s = 0;
#pragma unroll
            for(int q = 0; q < kItems; ++q) {
                v[q] = b + q < n ? f[b + q] : 0u;
                s += v[q] ? 1u : 0u;
                cells += v[q];
            }
            uint32_t total, at = 0;
            at = carry + block_exclusive_scan(s, sh, total);
#pragma unroll
            for(int q = 0; q < kItems; ++q)
                if(b + q < n) {
                    brickSlot[l][b + q] = v[q] ? (int32_t)at : -1;
                    if(v[q]) {
                        slotBrick[l][at++] = (int32_t)(b + q);
                        if(l) f[b + q] = 0;
                    }
                }
            carry += total;
        }
        uint32_t total;
        block_exclusive_scan(cells, sh, total);
        if(threadIdx.x == 0) {
            out[1 + l] = carry;
            if(l == 0) out[0] = total;
        }
    }
};

// The active bricks' tables, all levels in one launch. nbr: the six neighbours' slots (-x, +x, -y, +y, -z,
// +z; -1: none). ptab (8 ints, not on the coarsest level): the coarse bricks that a brick's cells and halo
// can have as parents, its own parent's six neighbours and (index 6) the parent; then the parities of the
// brick's coordinates.
struct k_brick_tables {
    static constexpr int kThreads = kBlock;
    int            nLevels;
    uint32_t       first[kMaxMgLevels], nSlots[kMaxMgLevels];  // first block
    int            nbx[kMaxMgLevels], nby[kMaxMgLevels], nbz[kMaxMgLevels];
    const int32_t *brickSlot[kMaxMgLevels], *slotBrick[kMaxMgLevels];
    int32_t *      nbr[kMaxMgLevels], *ptab[kMaxMgLevels];
    __device__ void operator()(Blk blk) const {
        int l = 0;
        while(l + 1 < nLevels && blk.id >= first[l + 1]) ++l;
        const uint32_t s = (blk.id - first[l]) * blockDim.x + threadIdx.x;
        if(s >= nSlots[l]) return;
        const int b = slotBrick[l][s], bx = b % nbx[l], by = (b / nbx[l]) % nby[l], bz = b / (nbx[l] * nby[l]);
        auto      slots = [&](int m, int x, int y, int z, int32_t* out) {
            const int       X = nbx[m], Y = nby[m], Z = nbz[m];
            const int32_t * t = brickSlot[m], o = (z * Y + y) * X + x;
            out[0] = x > 0 ? t[o - 1] : -1;
            out[1] = x + 1 < X ? t[o + 1] : -1;
            out[2] = y > 0 ? t[o - X] : -1;
            out[3] = y + 1 < Y ? t[o + X] : -1;
            out[4] = z > 0 ? t[o - X * Y] : -1;
            out[5] = z + 1 < Z ? t[o + X * Y] : -1;
        };
        slots(l, bx, by, bz, nbr[l] + 6 * s);
        if(l + 1 < nLevels) {
            int32_t* t = ptab[l] + 8 * s;
            slots(l + 1, bx >> 1, by >> 1, bz >> 1, t);
            t[6] = brickSlot[l + 1][((bz >> 1) * nby[l + 1] + (by >> 1)) * nbx[l + 1] + (bx >> 1)];
            t[7] = (bx & 1) | (by & 1) << 1 | (bz & 1) << 2;
        }
    }
};

// vector index of the neighbour of local cell l in direction dir (-1 when absent)
__device__ __forceinline__ int32_t nbr_index(const int32_t* __restrict__ nbr, int32_t s, int l, int dir) {
    const int lx = l & 7, ly = (l >> 3) & 7, lz = l >> 6;
    switch(dir) {
        case 0: return lx > 0 ? s * 512 + l - 1 : (nbr[6 * s + 0] >= 0 ? nbr[6 * s + 0] * 512 + l + 7 : -1);
        case 1: return lx < 7 ? s * 512 + l + 1 : (nbr[6 * s + 1] >= 0 ? nbr[6 * s + 1] * 512 + l - 7 : -1);
        case 2: return ly > 0 ? s * 512 + l - 8 : (nbr[6 * s + 2] >= 0 ? nbr[6 * s + 2] * 512 + l + 56 : -1);
        case 3: return ly < 7 ? s * 512 + l + 8 : (nbr[6 * s + 3] >= 0 ? nbr[6 * s + 3] * 512 + l - 56 : -1);
        case 4: return lz > 0 ? s * 512 + l - 64 : (nbr[6 * s + 4] >= 0 ? nbr[6 * s + 4] * 512 + l + 448 : -1);
        default: return lz < 7 ? s * 512 + l + 64 : (nbr[6 * s + 5] >= 0 ? nbr[6 * s + 5] * 512 + l - 448 : -1);
    }
}

//==================================================================================================
// computeSystem (PIC_Solver.cpp:693-893), matrix-free form. Per fluid interior cell: rhs (FP64,
// negative divergence), diagonal and the +x/+y/+z couplings (-w*dt when both cells are fluid), in
// FP64 and rounded to FP32. Cells outside [1, n-2] keep an empty row, as in the reference.
//==================================================================================================
struct SystemOut {
    double *rhs64, *diag64, *cx64, *cy64, *cz64;  // cx64..: may be null (FP32 mode)
    float * rhs32, *diag32, *cx32, *cy32, *cz32, *invdiag32;
    int32_t* uni;  // per brick: see UniformRow
};

// A brick deep in the fluid has the same row in all its 512 cells: six fluid neighbours through fully open
// faces, so every coupling is -dt and the diagonal 6 dt as the assembly sums it. k_assemble flags such
// bricks, and the kernels that stream the finest level take the row from here instead of reading it: 4 of
// 8 words a cell of the SpMV, 32 of 52 bytes of the FP64 residual. Same values, same bits. At 256^3 (9593
// bricks, about 60% of them uniform): SpMV 33.7 -> 28.5 us, update 35.2 -> 32.6, restriction 24.1 -> 19.8,
// post-smoother 47.0 -> 44.5, FP64 residual 70.3 -> 49.0. The flag comes before the row in a dependent chain,
// 0.5 us of the 4.6 us an SpMV of 216 bricks takes, so small systems have nothing to gain: refined projections
// of full boxes of 216 to 1000 bricks take the same time with and without, within the runs' 2%; of 1331 bricks
// 2210 -> 2165 us, 2197 2850 -> 2770, 8000 5850 -> 5540. Up to kUniformMin bricks every row is read.
constexpr uint32_t kUniformMin = 1024;

struct UniformRow {
    const int32_t* flag;  // per brick; null: none
    double c64, d64;
    float  c, d, inv;
    UniformRow() = default;
    UniformRow(const int32_t* f, float dt) : flag(f) {
        const double t = (double)dt;
        c64 = -t;
        d64 = ((((t + t) + t) + t) + t) + t;
        c   = (float)c64;
        d   = (float)d64;
        inv = d64 > 0 ? (float)(1.0 / d64) : 0.f;  // as k_assemble: a projection may be given any time step
    }
    __device__ __forceinline__ bool is(int s) const { return flag && flag[s] != 0; }
};

struct k_assemble {
    static constexpr int kThreads = 512;
    const int32_t* __restrict__ slotBrick;
    GridGeom g;
    const float* __restrict__ phi;
    VelGrid G;
    const float* __restrict__ wu;
    const float* __restrict__ wv;
    const float* __restrict__ ww;
    float dt;
    SystemOut S;
    __device__ void operator()(Blk blk) const {
        const int s = blk.id, l = threadIdx.x;
        const int b = slotBrick[s];
        const int bx = b % g.nbx, by = (b / g.nbx) % g.nby, bz = b / (g.nbx * g.nby);
        const int i = bx * 8 + (l & 7), j = by * 8 + ((l >> 3) & 7), k = bz * 8 + (l >> 6);
        const size_t o = (size_t)s * 512 + l;
        double rhs = 0, diag = 0, cx = 0, cy = 0, cz = 0;
        int    same = 0;  // the uniform row
        const bool interior = i >= 1 && j >= 1 && k >= 1 && i <= g.nx - 2 && j <= g.ny - 2 && k <= g.nz - 2;
        if(interior) {
            auto P = [&](int a, int c, int e) { return phi[lin3(a, c, e, g.nx, g.ny)]; };
            const float pc = P(i, j, k);
            if(pc < 0) {
                const int    ux = g.nx + 1, vy = g.ny + 1;
                const double wr = wu[lin3(i + 1, j, k, ux, g.ny)], wl = wu[lin3(i, j, k, ux, g.ny)];
                const double wt = wv[lin3(i, j + 1, k, g.nx, vy)], wb = wv[lin3(i, j, k, g.nx, vy)];
                const double wf = ww[lin3(i, j, k + 1, g.nx, g.ny)], wn = ww[lin3(i, j, k, g.nx, g.ny)];
                rhs -= wr * (double)G.u[lin3(i + 1, j, k, ux, g.ny)];
                rhs += wl * (double)G.u[lin3(i, j, k, ux, g.ny)];
                rhs -= wt * (double)G.v[lin3(i, j + 1, k, g.nx, vy)];
                rhs += wb * (double)G.v[lin3(i, j, k, g.nx, vy)];
                rhs -= wf * (double)G.w[lin3(i, j, k + 1, g.nx, g.ny)];
                rhs += wn * (double)G.w[lin3(i, j, k, g.nx, g.ny)];
                const double ddt = (double)dt;
                const double pcd = (double)pc;
                auto side = [&](float pn, double w, double& coupling, bool upper) {
                    const double term = w * ddt;
                    if(pn < 0) {
                        diag += term;
                        if(upper) coupling = -term;
                    } else {
                        const double th = fraction_inside2(pcd, (double)pn);
                        diag += term / (th > 0.01 ? th : 0.01);
                    }
                };
                double dummy = 0;
                side(P(i + 1, j, k), wr, cx, true);
                side(P(i - 1, j, k), wl, dummy, false);
                side(P(i, j + 1, k), wt, cy, true);
                side(P(i, j - 1, k), wb, dummy, false);
                side(P(i, j, k + 1), wf, cz, true);
                side(P(i, j, k - 1), wn, dummy, false);
                same = wr == 1 && wl == 1 && wt == 1 && wb == 1 && wf == 1 && wn == 1 && P(i + 1, j, k) < 0 && P(i - 1, j, k) < 0 &&
                       P(i, j + 1, k) < 0 && P(i, j - 1, k) < 0 && P(i, j, k + 1) < 0 && P(i, j, k - 1) < 0 && i + 1 <= g.nx - 2 &&
                       j + 1 <= g.ny - 2 && k + 1 <= g.nz - 2 && i >= 2 && j >= 2 && k >= 2;
                // couplings into boundary-layer cells (empty rows) are dropped
                if(i + 1 > g.nx - 2) cx = 0;
                if(j + 1 > g.ny - 2) cy = 0;
                if(k + 1 > g.nz - 2) cz = 0;
            }
        }
        if(S.rhs64) S.rhs64[o] = rhs;
        if(S.diag64) {
            S.diag64[o] = diag;
            S.cx64[o]   = cx;
            S.cy64[o]   = cy;
            S.cz64[o]   = cz;
        }
        S.rhs32[o]     = (float)rhs;
        S.diag32[o]    = (float)diag;
        S.cx32[o]      = (float)cx;
        S.cy32[o]      = (float)cy;
        S.cz32[o]      = (float)cz;
        S.invdiag32[o] = diag > 0 ? (float)(1.0 / diag) : 0.f;
        same           = __syncthreads_and(same);
        if(l == 0) S.uni[s] = same ? 1 : 0;
    }
};

//==================================================================================================
// PCG (PCGSolver.cpp:143-199) with Jacobi preconditioning, FP32 vectors and FP64 scalars.
// Scalars and the stop flag live in device memory; every kernel returns at once after the stop
// flag is set, so the host can queue iterations in chunks without reading back per iteration.
// Reductions: per-block partials, then a one-block kernel folds them in fixed order.
//==================================================================================================
struct PcgState {
    double   rho, alpha, beta, tmp;
    float    tol, res, bmax, pad0;
    uint32_t iter, maxIter, done, success;
};

// Reductions are two-level and deterministic: each block of a main kernel reduces a fixed set of
// bricks (b, b + the block count, ... or a contiguous chunk) and writes one partial with a plain store; a
// one-block fold kernel then combines the partials in index order. Kernel boundaries order the two,
// so no device-scope fences are needed inside the main kernels.
constexpr int kMaxRedBlocks = 2048;

template<int NT> __device__ __forceinline__ double block_sum(double v, double* sh) {
    v = wave_sum(v);
    if((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    if(threadIdx.x == 0)
        for(int i = 0; i < NT / 64; ++i) t += sh[i];
    __syncthreads();
    return t;  // valid in thread 0
}
template<int NT> __device__ __forceinline__ double block_max(double v, double* sh) {
    v = wave_maxd(v);
    if((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    if(threadIdx.x == 0)
        for(int i = 0; i < NT / 64; ++i) t = fmax(t, sh[i]);
    __syncthreads();
    return t;
}

// fold n partials in fixed order (1024-thread block); sum (or max) valid in thread 0
__device__ __forceinline__ double fold(const double* __restrict__ p, int n, bool isMax, double* sh) {
    double a = 0;
    for(int i = threadIdx.x; i < n; i += 1024) a = isMax ? fmax(a, p[i]) : a + p[i];
    return isMax ? block_max<1024>(a, sh) : block_sum<1024>(a, sh);
}

// The same sum by every workgroup of a consumer kernel (NT threads), for n <= kFoldMax partials: valid
// in all threads and, with fold()'s order (64 consecutive partials per wavefront sum, then the sums in
// order), the same bits; sh holds kFoldMax / 64 sums. On small systems it replaces a one-block launch
// (2.5-3.5 us of an iteration of about 90 at 64^3). Refined projections with the launch and without it: 216
// bricks 1510 -> 1440 us, 512 1770 -> 1690, 729 2170 -> 2100, 1000 2280 -> 2240. With more partials every
// workgroup's fold costs more than the launch: 1331 bricks 2230 -> 2310 us, 1728 2490 -> 2730.
constexpr int kFoldMax = 1024;
template<int NT> __device__ __forceinline__ double fold_all(const double* __restrict__ p, int n, double* sh) {
    double v[kFoldMax / NT];
#pragma unroll
    for(int k = 0; k < kFoldMax / NT; ++k) {
        const int i = k * NT + (int)threadIdx.x;
        v[k]        = 0.0;
        if(k * NT < n) v[k] = i < n ? p[i] : 0.0;
    }
#pragma unroll
    for(int k = 0; k < kFoldMax / NT; ++k)
        if(k * NT < n) {
            const double s = wave_sum(v[k]);
            if((threadIdx.x & 63) == 0) sh[k * (NT / 64) + (threadIdx.x >> 6)] = s;
        }
    __syncthreads();
    double    t = 0;
    const int m = (n + NT - 1) / NT * (NT / 64);
    for(int w = 0; w < m; ++w) t += sh[w];
    __syncthreads();
    return t;
}

// max|r| of an iteration where the restriction needs it at once (the multigrid's fused update): 64 words, a
// cache line each, that take the bricks' maxima by atomicMax on the bits of non-negative floats, which no
// order changes. The SpMV before clears them. A fold of the bricks' partials took a launch of its own (2.4 us
// at 1309 bricks, 4.6 at 9593, and the gap before the next) or, on small systems, reads in every workgroup
// of the restriction (4.6 us at 216 bricks, now 4.3).
constexpr int kMaxWords = 64, kMaxWordStep = 32;
__device__ __forceinline__ void max_words_clear(uint32_t* w, Blk blk) {
    if(w && blk.id == 0 && threadIdx.x < kMaxWords) w[kMaxWordStep * threadIdx.x] = 0u;
}
__device__ __forceinline__ void  max_words_put(uint32_t* w, uint32_t brick, float m) { atomicMax(w + kMaxWordStep * (brick % kMaxWords), __float_as_uint(m)); }

// the stop test of an iteration (PCGSolver.cpp:182-187), B = max|r|. With the multigrid preconditioner it
// runs before the V-cycle: the last iteration of a solve needs none (two thirds of an iteration's time, and
// a solve has 5 to 10 iterations).
__device__ __forceinline__ void pcg_stop_test(PcgState& st, double B) {
    st.iter += 1;
    st.res = (float)B;
    if((float)B < st.tol) {
        st.done    = 1;
        st.success = 1;
    } else if(st.iter >= st.maxIter) {
        st.done = 1;
    }
}
// init: x = 0, r = b, s = 0, z = M^-1 r; partials of z.r and max|b|
struct k_pcg_init {
    static constexpr int kThreads = 512;
    const float* __restrict__ b;
    const float* __restrict__ invdiag;
    float* __restrict__ x;
    float* __restrict__ r;
    float* __restrict__ z;
    float* __restrict__ s;
    uint32_t nSlots;
    double* __restrict__ pa;
    double* __restrict__ pb;
    int jacobi;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[8];
        double            rz = 0, m = 0;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const size_t o  = (size_t)slot * 512 + threadIdx.x;
            const float  bv = b[o];
            x[o]            = 0.f;
            r[o]            = bv;
            s[o]            = 0.f;
            if(jacobi) {
                const float zv = invdiag[o] * bv;
                z[o]           = zv;
                rz += (double)zv * (double)bv;
            }
            m = fmax(m, (double)fabsf(bv));
        }
        if(jacobi) rz = block_sum<512>(rz, sh);
        m = block_max<512>(m, sh);
        if(threadIdx.x == 0) {
            if(jacobi) pa[blk.id] = rz;
            pb[blk.id] = m;
        }
    }
};

// pa: na partials of z.r, pb: nb partials of max|b|
struct k_pcg_init_fin {
    static constexpr int kThreads = 1024;
    PcgState* st;
    const double* __restrict__ pa;
    int na;
    const double* __restrict__ pb;
    int nb;
    float relTol;
    uint32_t maxIter;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[16];
        const double      A = fold(pa, na, false, sh);
        const double      B = fold(pb, nb, true, sh);
        if(threadIdx.x != 0) return;
        st->bmax    = (float)B;
        st->res     = (float)B;
        st->iter    = 0;
        st->maxIter = maxIter;
        st->beta    = 0;
        st->rho     = A;
        st->done    = 0;
        st->success = 0;
        st->tol     = relTol * (float)B;  // PCGSolver.cpp:160
        if((float)B < kFltMin) {          // PCGSolver.cpp:155-158
            st->done    = 1;
            st->success = 1;
        } else if(A < (double)kFltMin || isnan(A)) {  // PCGSolver.cpp:164-167
            st->done = 1;
        } else if(maxIter == 0) {
            st->done = 1;
        }
    }
};

// s_out = z + beta s_in ; q = A s_out ; partial s_out . q
// the slots of this block when the grid shares n slots: one contiguous chunk per block, and the
// chunks of one XCD's blocks (equal block index mod 8) adjacent, so that brick faces read from
// neighbouring bricks are mostly in that XCD's L2
__device__ __forceinline__ void block_chunk(Blk blk, uint32_t n, uint32_t& s0, uint32_t& s1) {
    const uint32_t G = blk.n, b = blk.id, xcd = b % 8u, q = G / 8u, r = G % 8u;
    const uint32_t v = xcd * q + min(xcd, r) + b / 8u;
    s0               = (uint32_t)(((uint64_t)n * v) / G);
    s1               = (uint32_t)(((uint64_t)n * (v + 1)) / G);
}

// kFold (small systems): the last iteration's beta (k_pcg_beta) is formed here, from st to the other
// state `next` (null: it has been), over nPart <= kFoldMax partials rz of z.r
template<bool kFold>
struct k_pcg_spmv {
    static constexpr int kThreads = 512;
    const int32_t* __restrict__ nbr;
    const float* __restrict__ z;
    const float* __restrict__ sin;
    float* __restrict__ sout;
    float* __restrict__ q;
    const float* __restrict__ diag;
    const float* __restrict__ cx;
    const float* __restrict__ cy;
    const float* __restrict__ cz;
    UniformRow uni;
    uint32_t nSlots;
    const PcgState* st;
    double* __restrict__ pa;
    PcgState* next;
    const double* __restrict__ rz;
    int nPart;
    uint32_t* maxWords;  // or null
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[kFoldMax / 64];
        float             beta;
        double            A = 0, be = 0;
        if(kFold && next) {
            const bool done = st->done != 0;
            A  = done ? 0.0 : fold_all<512>(rz, nPart, sh);
            be = A / st->rho;
            if(done) {
                if(blk.id == 0 && threadIdx.x == 0) *next = *st;
                return;
            }
            beta = (float)be;
        } else {
            if(st->done) return;
            beta = (float)st->beta;
        }
        const int   l    = threadIdx.x;
        double      d    = 0;
        uint32_t    s0, s1;
        block_chunk(blk, nSlots, s0, s1);
        for(uint32_t slot = s0; slot < s1; ++slot) {
            const int     s   = (int)slot;
            const size_t  o   = (size_t)s * 512 + l;
            auto          S   = [&](int32_t idx) { return z[idx] + beta * sin[idx]; };
            const float   sc  = z[o] + beta * sin[o];
            const int32_t ixm = nbr_index(nbr, s, l, 0), ixp = nbr_index(nbr, s, l, 1);
            const int32_t iym = nbr_index(nbr, s, l, 2), iyp = nbr_index(nbr, s, l, 3);
            const int32_t izm = nbr_index(nbr, s, l, 4), izp = nbr_index(nbr, s, l, 5);
            // a missing neighbour reads the cell itself with a zero coupling (adds exactly nothing), so
            // all loads are unconditional
            const int32_t oi = (int32_t)o;
            const int32_t jxm = ixm >= 0 ? ixm : oi, jxp = ixp >= 0 ? ixp : oi, jym = iym >= 0 ? iym : oi;
            const int32_t jyp = iyp >= 0 ? iyp : oi, jzm = izm >= 0 ? izm : oi, jzp = izp >= 0 ? izp : oi;
            float czm = uni.c, cym = uni.c, cxm = uni.c, cxp = uni.c, cyp = uni.c, czp = uni.c, dia = uni.d;
            if(!uni.is(s)) {
                czm = cz[jzm];
                cym = cy[jym];
                cxm = cx[jxm];
                cxp = cx[o];
                cyp = cy[o];
                czp = cz[o];
                dia = diag[o];
            }
            const float   szm = S(jzm), sym = S(jym), sxm = S(jxm), sxp = S(jxp), syp = S(jyp), szp = S(jzp);
            float         acc = 0.f;
            acc += (izm >= 0 ? czm : 0.f) * szm;
            acc += (iym >= 0 ? cym : 0.f) * sym;
            acc += (ixm >= 0 ? cxm : 0.f) * sxm;
            acc += dia * sc;
            acc += (ixp >= 0 ? cxp : 0.f) * sxp;
            acc += (iyp >= 0 ? cyp : 0.f) * syp;
            acc += (izp >= 0 ? czp : 0.f) * szp;
            sout[o] = sc;
            q[o]    = acc;
            d += (double)sc * (double)acc;
        }
        d = block_sum<512>(d, sh);
        if(threadIdx.x == 0) pa[blk.id] = d;
        // stores to the state come last (see k_mg_residual_restrict)
        max_words_clear(maxWords, blk);
        if(kFold && next && blk.id == 0 && threadIdx.x == 0) {
            *next      = *st;
            next->beta = be;
            next->rho  = A;
        }
    }
};

// tmp = s.q ; alpha = rho / tmp (PCGSolver.cpp:174-180)
struct k_pcg_alpha {
    static constexpr int kThreads = 1024;
    PcgState* st;
    const double* __restrict__ pa;
    int n;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[16];
        if(st && st->done) return;
        const double A = fold(pa, n, false, sh);
        if(threadIdx.x != 0) return;
        st->tmp = A;
        if(A < (double)kFltMin) {
            st->done    = 1;
            st->success = 1;
            st->iter += 1;
        } else {
            st->alpha = st->rho / A;
        }
    }
};

// x += alpha s ; r -= alpha q ; z = M^-1 r ; partials z.r and max|r|
struct k_pcg_update {
    static constexpr int kThreads = 512;
    const float* __restrict__ s;
    const float* __restrict__ q;
    const float* __restrict__ invdiag;
    float* __restrict__ x;
    float* __restrict__ r;
    float* __restrict__ z;
    uint32_t nSlots;
    const PcgState* __restrict__ st;
    double* __restrict__ pa;
    double* __restrict__ pb;
    int jacobi;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[8];
        if(st && st->done) return;
        const float alpha = (float)st->alpha;
        double      rz = 0, m = 0;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const size_t o  = (size_t)slot * 512 + threadIdx.x;
            const float  xv = x[o] + alpha * s[o];
            const float  rv = r[o] + (-alpha) * q[o];
            x[o]            = xv;
            r[o]            = rv;
            if(jacobi) {  // z = M^-1 r fused here; the multigrid preconditioner runs after this kernel
                const float zv = invdiag[o] * rv;
                z[o]           = zv;
                rz += (double)zv * (double)rv;
            }
            m = fmax(m, (double)fabsf(rv));
        }
        if(jacobi) rz = block_sum<512>(rz, sh);
        m = block_max<512>(m, sh);
        if(threadIdx.x == 0) {
            if(jacobi) pa[blk.id] = rz;
            pb[blk.id] = m;
        }
    }
};

// res = max|r| from nb partials pb and the stop test (PCGSolver.cpp:182-187), when pb is given; then beta =
// rz / rho (:190-194) from na partials pa of z.r, when pa is given
struct k_pcg_beta {
    static constexpr int kThreads = 1024;
    PcgState* st;
    const double* __restrict__ pa;
    int na;
    const double* __restrict__ pb;
    int nb;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[16];
        if(st && st->done) return;
        const double A = pa ? fold(pa, na, false, sh) : 0.0;
        const double B = pb ? fold(pb, nb, true, sh) : 0.0;
        if(threadIdx.x != 0) return;
        if(pb) pcg_stop_test(*st, B);
        if(pa && !st->done) {
            st->beta = A / st->rho;
            st->rho  = A;
        }
    }
};

//--------------------------------------------------------------------------------------------------
// FP64 defect correction: r64 = b64 - A64 x64, max|r64|, max|b64|, r32 = (float) r64 (inner rhs)
//--------------------------------------------------------------------------------------------------
struct OuterState {
    double res, bmax;
};
// what the host reads back of a solve: the inner solve's two states and the outer one's
struct SolveState {
    PcgState   inner[2];
    OuterState outer;
};
// The end of an outer pass (accumulate, next residual) can be queued behind the inner iterations before the
// host knows that they suffice: with a gate it runs only when the inner solve has stopped.
__device__ __forceinline__ bool gated(const PcgState* gate) { return gate && !gate->done; }

struct k_residual64 {
    static constexpr int kThreads = 512;
    const int32_t* __restrict__ nbr;
    const double* __restrict__ x;
    const double* __restrict__ b;
    const double* __restrict__ diag;
    const double* __restrict__ cx;
    const double* __restrict__ cy;
    const double* __restrict__ cz;
    UniformRow uni;
    float* __restrict__ r32;
    uint32_t nSlots;
    double* __restrict__ pa;
    double* __restrict__ pb;
    int first;
    const PcgState* gate;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[8];
        if(gated(gate)) return;
        const int         l = threadIdx.x;
        double            m = 0, bm = 0;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const int    s  = (int)slot;
            const size_t o  = (size_t)s * 512 + l;
            double       ax = 0.0;
            if(!first && uni.is(s)) {  // every neighbour is there
                ax += uni.c64 * x[nbr_index(nbr, s, l, 4)];
                ax += uni.c64 * x[nbr_index(nbr, s, l, 2)];
                ax += uni.c64 * x[nbr_index(nbr, s, l, 0)];
                ax += uni.d64 * x[o];
                ax += uni.c64 * x[nbr_index(nbr, s, l, 1)];
                ax += uni.c64 * x[nbr_index(nbr, s, l, 3)];
                ax += uni.c64 * x[nbr_index(nbr, s, l, 5)];
            } else if(!first) {
                const int32_t ixm = nbr_index(nbr, s, l, 0), ixp = nbr_index(nbr, s, l, 1);
                const int32_t iym = nbr_index(nbr, s, l, 2), iyp = nbr_index(nbr, s, l, 3);
                const int32_t izm = nbr_index(nbr, s, l, 4), izp = nbr_index(nbr, s, l, 5);
                if(izm >= 0) ax += cz[izm] * x[izm];
                if(iym >= 0) ax += cy[iym] * x[iym];
                if(ixm >= 0) ax += cx[ixm] * x[ixm];
                ax += diag[o] * x[o];
                if(ixp >= 0) ax += cx[o] * x[ixp];
                if(iyp >= 0) ax += cy[o] * x[iyp];
                if(izp >= 0) ax += cz[o] * x[izp];
            }
            const double bv = b[o];
            const double rv = bv - ax;
            r32[o]          = (float)rv;
            m               = fmax(m, fabs(rv));
            bm              = fmax(bm, fabs(bv));
        }
        m  = block_max<512>(m, sh);
        bm = block_max<512>(bm, sh);
        if(threadIdx.x == 0) {
            pa[blk.id] = m;
            pb[blk.id] = bm;
        }
    }
};

struct k_residual64_fin {
    static constexpr int kThreads = 1024;
    OuterState* ost;
    const double* __restrict__ pa;
    const double* __restrict__ pb;
    int n;
    const PcgState* gate;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[16];
        if(gated(gate)) return;
        const double      M  = fold(pa, n, true, sh);
        const double      BM = fold(pb, n, true, sh);
        if(threadIdx.x == 0) {
            ost->res  = M;
            ost->bmax = BM;
        }
    }
};

// the previous solve's pressure as the initial guess of the next refined solve: cell l of new slot s
// takes the old value of the same cell when it is fluid now (phi < 0) and its brick had a slot then
// (prevBrickSlot: the old brick -> slot table), else 0
struct k_warm_start {
    static constexpr int kThreads = 512;
    const int32_t* __restrict__ slotBrick;
    const int32_t* __restrict__ prevBrickSlot;
    const double* __restrict__  xprev;
    const float* __restrict__   phi;
    GridGeom                    g;
    uint32_t                    nSlots;
    double* __restrict__        x;
    __device__ void operator()(Blk blk) const {
        const int l = threadIdx.x;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const int32_t b  = slotBrick[slot];
            const int32_t os = prevBrickSlot[b];
            const int     bx = b % g.nbx, by = (b / g.nbx) % g.nby, bz = b / (g.nbx * g.nby);
            const int     i = bx * 8 + (l & 7), j = by * 8 + ((l >> 3) & 7), k = bz * 8 + (l >> 6);
            const bool    fluid = i < g.nx && j < g.ny && k < g.nz && phi[lin3(i, j, k, g.nx, g.ny)] < 0.f;
            x[(size_t)slot * 512 + l] = (fluid && os >= 0) ? xprev[(size_t)os * 512 + l] : 0.0;
        }
    }
};

struct k_accumulate64 {
    static constexpr int kThreads = 512;
    double* __restrict__ x64;
    const float* __restrict__ d;
    uint32_t nSlots;
    int first;
    const PcgState* gate;
    __device__ void operator()(Blk blk) const {
        if(gated(gate)) return;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const size_t o = (size_t)slot * 512 + threadIdx.x;
            x64[o]         = first ? (double)d[o] : x64[o] + (double)d[o];
        }
    }
};

//==================================================================================================
// updateProjectedVelocity (PIC_Solver.cpp:911-981), one thread per face; faces the reference does
// not update are zeroed with valid = 0 (its serial pass, :973-980)
//==================================================================================================
template<class PT> struct PressView {
    const PT*      x;
    const int32_t* brickSlot;
};

template<class PT> __device__ __forceinline__ PT pressure_at(const PressView<PT>& pv, const GridGeom& g, int i, int j, int k) {
    const int32_t s = pv.brickSlot[((k >> 3) * g.nby + (j >> 3)) * g.nbx + (i >> 3)];
    return pv.x[(size_t)s * 512 + ((k & 7) * 8 + (j & 7)) * 8 + (i & 7)];
}

// The three components in one launch, four faces a thread: where no fluid cell touches the four (three
// quarters of the grid at 256^3), velocities and weights are not even read. 326 -> 243 us there.
template<class PT>
struct k_update_velocity {
    static constexpr int kThreads = kBlock;
    float*         vel[3];
    uint8_t*       valid[3];
    const float*   weight[3];
    uint32_t       n[3], first[3];  // faces, first block
    const float* __restrict__ phi;
    PressView<PT> pv;
    GridGeom g;
    float dt;
    static uint32_t blocks(uint32_t n) { return (n + 4 * kThreads - 1) / (4 * kThreads); }
    __device__ void operator()(Blk blk) const {
        const int      d  = blk.id >= first[2] ? 2 : (blk.id >= first[1] ? 1 : 0);
        const uint32_t t0 = 4u * ((blk.id - first[d]) * kThreads + threadIdx.x), N = n[d];
        if(t0 >= N) return;
        const int sx = g.nx + (d == 0), sy = g.ny + (d == 1), m = (int)min(4u, N - t0);
        const int an = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
        const uint32_t back = d == 0 ? 1u : (d == 1 ? (uint32_t)g.nx : (uint32_t)g.nx * (uint32_t)g.ny);  // to the cell before the face
        int   i[4], j[4], k[4];
        float pc[4], pl[4];
        bool  fluid[4], any = false;
        unlin3(t0, sx, sy, i[0], j[0], k[0]);
#pragma unroll
        for(int q = 1; q < 4; ++q) {  // along x, into the next row where it ends
            const bool row = i[q - 1] + 1 == sx, slab = row && j[q - 1] + 1 == sy;
            i[q] = row ? 0 : i[q - 1] + 1;
            j[q] = slab ? 0 : j[q - 1] + (row ? 1 : 0);
            k[q] = k[q - 1] + (slab ? 1 : 0);
        }
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            const int ai = d == 0 ? i[q] : (d == 1 ? j[q] : k[q]);  // index along the face normal
            pc[q] = pl[q] = 0.f;
            if(q < m && ai > 0 && ai < an) {
                const uint32_t c = (uint32_t)lin3(i[q], j[q], k[q], g.nx, g.ny);
                pc[q]            = phi[c];
                pl[q]            = phi[c - back];
            }
        }
#pragma unroll
        for(int q = 0; q < 4; ++q) any |= fluid[q] = pc[q] < 0 || pl[q] < 0;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        uint8_t ok[4] = {0, 0, 0, 0};
        if(any) {
#pragma unroll
            for(int q = 0; q < 4; ++q)
                if(fluid[q] && weight[d][t0 + q] > 0.f) {
                    const PT prc = pc[q] < 0 ? pressure_at(pv, g, i[q], j[q], k[q]) : PT(0);
                    const PT prl = pl[q] < 0 ? pressure_at(pv, g, i[q] - (d == 0), j[q] - (d == 1), k[q] - (d == 2)) : PT(0);
                    PT       th  = fraction_inside2((PT)pl[q], (PT)pc[q]);
                    th           = th > PT(0.01) ? th : PT(0.01);  // std::max(0.01, th)
                    v[q]         = (float)((PT)vel[d][t0 + q] - (PT)dt * (prc - prl) / th);
                    ok[q]        = 1;
                }
        }
        if(m == 4) {
            *reinterpret_cast<float4*>(vel[d] + t0)   = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<uchar4*>(valid[d] + t0) = make_uchar4(ok[0], ok[1], ok[2], ok[3]);
        } else {
            for(int q = 0; q < m; ++q) {
                vel[d][t0 + q]   = v[q];
                valid[d][t0 + q] = ok[q];
            }
        }
    }
};

//==================================================================================================
// mapGrid2Particles with the FLIP blend (FLIP_Solver.cpp:99-133, MathHelpers.h:549-551). Bound by the
// vector memory instructions of the gathers: each grid's stencil is loaded once, for the value and the
// change (28 loads a wavefront where the two interpolations issued 41): 801 -> 576 us for 33M particles
// at 256^3; AFLIP, 1.7M: 84 -> 59 us.
//==================================================================================================
struct OldGrid {
    const float *u, *v, *w;
};

struct k_g2p {
    static constexpr int kThreads = kBlock;
    Particles P;
    uint32_t n;
    VelGrid G;
    OldGrid O;
    GridGeom g;
    float ratio;
    __device__ void operator()(Blk blk) const {
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        if(p >= n) return;
        const float4 gq = P.gp[p];
        const float  a  = 1.0f - ratio;
        auto         blend = [&](const float* __restrict__ n, const float* __restrict__ o, const Stencil& s, float v) {
            const Corners c = corners(n, s), d = corner_diff(c, corners(o, s));
            return a * interp8(c, s) + ratio * (v + interp8(d, s));
        };
        const float vx = blend(G.u, O.u, stencil3(g.nx + 1, g.ny, g.nz, gq.x, gq.y - 0.5f, gq.z - 0.5f), P.vx[p]);
        const float vy = blend(G.v, O.v, stencil3(g.nx, g.ny + 1, g.nz, gq.x - 0.5f, gq.y, gq.z - 0.5f), P.vy[p]);
        const float vz = blend(G.w, O.w, stencil3(g.nx, g.ny, g.nz + 1, gq.x - 0.5f, gq.y - 0.5f, gq.z), P.vz[p]);
        P.vx[p] = vx;
        P.vy[p] = vy;
        P.vz[p] = vz;
    }
};

//==================================================================================================
// APIC / AFLIP (APIC_Solver.cpp:42-125, AFLIP_Solver.cpp:43-140): each particle carries an affine
// matrix C (row d = the gradient of velocity component d), stored as nine arrays in the particles'
// storage order and moved with them by the binning permute.
//==================================================================================================
struct k_permute_affine {
    static constexpr int kThreads = kBlock;
    Affine in;
    Affine out;
    const uint32_t* __restrict__ perm;
    uint32_t n;
    __device__ void operator()(Blk blk) const {
        const uint32_t i = blk.id * blockDim.x + threadIdx.x;
        if(i >= n) return;
        const uint32_t s = perm[i];
    #pragma unroll
        for(int k = 0; k < 9; ++k) out.c[k][i] = in.c[k][s];
    }
};

// APIC mapGrid2Particles (APIC_Solver.cpp:94-115): v = the interpolated grid velocity, C_d = the
// gradient of component d at gridPos - extra_d. AFLIP (AFLIP_Solver.cpp:94-140): both blended like
// FLIP, lerp(grid, particle + change, PIC_FLIP_ratio), the changes taken from vel - backup.
template<int kScheme>
struct k_g2p_affine {
    static constexpr int kThreads = kBlock;
    Particles P;
    Affine A;
    uint32_t n;
    VelGrid G;
    OldGrid O;
    GridGeom g;
    float ratio;
    __device__ void operator()(Blk blk) const {
    #pragma clang fp contract(off)
        const uint32_t p = blk.id * blockDim.x + threadIdx.x;
        if(p >= n) return;
        const float4 gq = P.gp[p];
        const float  a  = 1.0f - ratio;
        auto         gather = [&](const float* __restrict__ n, const float* __restrict__ o, const Stencil& s, float* v, float* const* m) {
            const Corners c = corners(n, s);
            float         gc[3];
            grad8(c, s, g.dx, gc);
            if(kScheme == 1) {
                v[p] = interp8(c, s);
#pragma unroll
                for(int k = 0; k < 3; ++k) m[k][p] = gc[k];
                return;
            }
            const Corners d = corner_diff(c, corners(o, s));
            float         dc[3];
            grad8(d, s, g.dx, dc);
            v[p] = a * interp8(c, s) + ratio * (v[p] + interp8(d, s));
#pragma unroll
            for(int k = 0; k < 3; ++k) m[k][p] = a * gc[k] + ratio * (m[k][p] + dc[k]);
        };
        gather(G.u, O.u, stencil3(g.nx + 1, g.ny, g.nz, gq.x, gq.y - 0.5f, gq.z - 0.5f), P.vx, A.c);
        gather(G.v, O.v, stencil3(g.nx, g.ny + 1, g.nz, gq.x - 0.5f, gq.y, gq.z - 0.5f), P.vy, A.c + 3);
        gather(G.w, O.w, stencil3(g.nx, g.ny, g.nz + 1, gq.x - 0.5f, gq.y - 0.5f, gq.z), P.vz, A.c + 6);
    }
};

// max |a| over the three components (timestepCFL, PIC_Solver.cpp:342-349); result via atomicMax on the bits.
// A launch reads all three, four values a load, and a workgroup whose maximum is no news leaves the result
// alone: 2048 atomics a component on the one word took 26 us each at 128^3, whatever the arrays' size; now
// 12.6 us for the three.
struct k_maxabs {
    static constexpr int kThreads = kBlock, kBlocks = 512;
    const float* a[3];
    uint32_t n[3];
    uint32_t* out;
    __device__ void operator()(Blk blk) const {
        __shared__ float sh[kBlock / 64];
        const uint32_t   t = blk.id * kBlock + threadIdx.x, T = blk.n * kBlock;
        float            m = 0.f;
        for(int c = 0; c < 3; ++c) {
            const float4* v = (const float4*)a[c];
            for(uint32_t i = t; i < n[c] / 4; i += T) {
                const float4 f = v[i];
                m = fmaxf(fmaxf(m, fmaxf(fabsf(f.x), fabsf(f.y))), fmaxf(fabsf(f.z), fabsf(f.w)));
            }
            if(t < n[c] % 4) m = fmaxf(m, fabsf(a[c][n[c] / 4 * 4 + t]));
        }
        m = wave_max(m);
        if((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
        __syncthreads();
        if(threadIdx.x == 0) {
            for(int i = 1; i < kBlock / 64; ++i) m = fmaxf(m, sh[i]);
            if(__float_as_uint(m) > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, __float_as_uint(m));
        }
    }
};

}  // namespace bnn

namespace bnn {

//==================================================================================================
// Multigrid preconditioner (extension; the reference's IC(0) is sequential). Level l+1 aggregates
// 2x2x2 cells of level l (piecewise-constant prolongation P); its operator is the Galerkin product
// P^T A P, which for a 7-point operator is again 7-point:
//   diag_C = sum_c diag_c + 2 * (couplings between children of C)
//   cxp_C  = sum of the 4 +x couplings leaving C's children with odd local x, etc.
// Every level stores 8^3-cell bricks (slot tables as on the fine level). The V-cycle is symmetric
// (red-black Gauss-Seidel: red then black before the coarse correction, black then red after), so
// M^-1 is symmetric positive definite and usable inside CG.
//==================================================================================================
struct LevelDev {
    int            nx, ny, nz, nbx, nby, nbz;
    const int32_t* brickSlot;
    const int32_t* slotBrick;
    const int32_t* nbr;
    const float *  diag, *cx, *cy, *cz, *invdiag;
    float *        x, *b, *r;
    uint32_t       nSlots;
    const int32_t* ptab;  // per slot: parent coarse brick and its six neighbours (8 ints), or null
    UniformRow     uni;   // finest level
};

__device__ __forceinline__ int32_t level_cell_index(const LevelDev& L, int i, int j, int k) {
    if(i < 0 || j < 0 || k < 0 || i >= L.nx || j >= L.ny || k >= L.nz) return -1;
    const int32_t s = L.brickSlot[((k >> 3) * L.nby + (j >> 3)) * L.nbx + (i >> 3)];
    return s < 0 ? -1 : s * 512 + ((k & 7) * 8 + (j & 7)) * 8 + (i & 7);
}

// Galerkin coefficients of the coarse level (one block per coarse brick, thread = coarse cell)
struct k_mg_coarsen {
    static constexpr int kThreads = 512;
    LevelDev F;
    LevelDev C;
    float* __restrict__ cdiag;
    float* __restrict__ ccx;
    float* __restrict__ ccy;
    float* __restrict__ ccz;
    float* __restrict__ cinv;
    float* __restrict__ cb;  // the right-hand side: the restriction writes only cells under an active fine brick
    __device__ void operator()(Blk blk) const {
        const int s = blk.id, l = threadIdx.x;
        const int b = C.slotBrick[s];
        const int bx = b % C.nbx, by = (b / C.nbx) % C.nby, bz = b / (C.nbx * C.nby);
        const int I = bx * 8 + (l & 7), J = by * 8 + ((l >> 3) & 7), K = bz * 8 + (l >> 6);
        float     d = 0.f, cx = 0.f, cy = 0.f, cz = 0.f, inner = 0.f;
        for(int c = 0; c < 8; ++c) {
            const int     a0 = c & 1, a1 = (c >> 1) & 1, a2 = (c >> 2) & 1;
            const int32_t f  = level_cell_index(F, 2 * I + a0, 2 * J + a1, 2 * K + a2);
            if(f < 0) continue;
            d += F.diag[f];
            if(a0) cx += F.cx[f];
            else inner += F.cx[f];
            if(a1) cy += F.cy[f];
            else inner += F.cy[f];
            if(a2) cz += F.cz[f];
            else inner += F.cz[f];
        }
        d += 2.f * inner;
        const size_t o = (size_t)s * 512 + l;
        cdiag[o]       = d;
        ccx[o]         = cx;
        ccy[o]         = cy;
        ccz[o]         = cz;
        cinv[o]        = d > 0.f ? 1.0f / d : 0.f;
        cb[o]          = 0.f;
    }
};

// sum of the six couplings times x. A missing neighbour reads the cell's own x (finite) with a zero
// coupling, which adds exactly nothing, so every load is issued before the first use.
__device__ __forceinline__ float level_offdiag_sum(const LevelDev& L, int s, int l, const float* __restrict__ x) {
    const int32_t ixm = nbr_index(L.nbr, s, l, 0), ixp = nbr_index(L.nbr, s, l, 1);
    const int32_t iym = nbr_index(L.nbr, s, l, 2), iyp = nbr_index(L.nbr, s, l, 3);
    const int32_t izm = nbr_index(L.nbr, s, l, 4), izp = nbr_index(L.nbr, s, l, 5);
    const int32_t o   = s * 512 + l;
    const int32_t jxm = ixm >= 0 ? ixm : o, jxp = ixp >= 0 ? ixp : o, jym = iym >= 0 ? iym : o;
    const int32_t jyp = iyp >= 0 ? iyp : o, jzm = izm >= 0 ? izm : o, jzp = izp >= 0 ? izp : o;
    const float   czm = L.cz[jzm], cym = L.cy[jym], cxm = L.cx[jxm], cxp = L.cx[o], cyp = L.cy[o], czp = L.cz[o];
    const float   xzm = x[jzm], xym = x[jym], xxm = x[jxm], xxp = x[jxp], xyp = x[jyp], xzp = x[jzp];
    float         acc = 0.f;
    acc += (izm >= 0 ? czm : 0.f) * xzm;
    acc += (iym >= 0 ? cym : 0.f) * xym;
    acc += (ixm >= 0 ? cxm : 0.f) * xxm;
    acc += (ixp >= 0 ? cxp : 0.f) * xxp;
    acc += (iyp >= 0 ? cyp : 0.f) * xyp;
    acc += (izp >= 0 ? czp : 0.f) * xzp;
    return acc;
}

__device__ __forceinline__ int cell_color(const LevelDev& L, int s, int l) {
    const int b = L.slotBrick[s];
    const int bx = b % L.nbx, by = (b / L.nbx) % L.nby, bz = b / (L.nbx * L.nby);
    return ((bx * 8 + (l & 7)) + (by * 8 + ((l >> 3) & 7)) + (bz * 8 + (l >> 6))) & 1;
}

// Launch order -> brick slot, a bijection on [0, n) that gives each XCD (the blocks with equal
// b % 8) one contiguous range of slots: slots are ordered by brick index, so a brick's neighbours,
// whose faces the stencils read, mostly sit in the same XCD's L2.
__device__ __forceinline__ uint32_t xcd_slot(uint32_t b, uint32_t n) {
    const uint32_t xcd = b % 8u, q = n / 8u, r = n % 8u;
    return xcd * q + min(xcd, r) + b / 8u;
}

// A brick's x with its one-cell halo in LDS (smoothers), x fastest. Rows of 12 and planes of 120 floats
// where 10 and 100 would do: a wave's accesses in a half-sweep (4 cells two apart in 8 rows of two planes)
// then fall on different banks, against two to a bank (a half-sweep of k_mg_tail over 8 bricks: 1110 ->
// 700 cycles).
constexpr int kTileRow = 12, kTilePlane = 120, kTile = 1200;
__device__ __forceinline__ int tile_index(int lx, int ly, int lz) { return (lz + 1) * kTilePlane + (ly + 1) * kTileRow + lx + 1; }

// The smoothers and the restriction work on pairs of cells: their loads, a cell each, were
// what bounded them (a load of 64 floats costs a CU 10 to 20 cycles however few bytes it moves; a pair takes
// half as many), and below some hundred bricks the steps from brick to parent in a launch. As pairs, with
// the parities and parents of the brick tables: at 216 / 9593 bricks update with pre-smoother 7.3 / 35.2 ->
// 5.8 / 31.9 us, restriction 6.4 / 18.6 -> 4.6 / 14.1 (before it took the stop test), post-smoother 6.9 / 33.7
// -> 6.0 / 33.3 (before it took the correction), the 64^3 step 1.90 -> 1.83 ms, 256^3 14.15 -> 13.85. (The
// SpMV, bound by latency and by the wavefronts in flight, lost as pairs: 27.8 -> 33.5 us.)

// The x-adjacent pair of cells that thread t of a brick's 256 owns, one of each colour: even is the first
// one's index in the brick, cr and cb the red (colour 0) and the black one's tile entries, offR the tile
// offset out of the pair from the red one (the black one's is -offR), swap: the first one is black.
struct BrickPair {
    int  px, ly, lz, even, cr, cb, offR;
    bool swap;
    __device__ __forceinline__ explicit BrickPair(int t) {
        px   = t & 3;
        ly   = (t >> 2) & 7;
        lz   = t >> 5;
        even = (lz * 8 + ly) * 8 + 2 * px;
        swap = (ly + lz) & 1;
        const int c = tile_index(2 * px, ly, lz);
        cr   = swap ? c + 1 : c;
        cb   = swap ? c : c + 1;
        offR = swap ? 1 : -1;
    }
    // the pair's parent in the parent brick, for a brick whose coordinates' parities are odd's bits
    __device__ __forceinline__ int parent(int odd) const {
        return (((odd >> 2 & 1) * 4 + lz / 2) * 8 + (odd >> 1 & 1) * 4 + ly / 2) * 8 + (odd & 1) * 4 + px;
    }
    __device__ __forceinline__ float red(float2 v) const { return swap ? v.y : v.x; }
    __device__ __forceinline__ float black(float2 v) const { return swap ? v.x : v.y; }
    __device__ __forceinline__ float2 cells(float r, float k) const { return swap ? make_float2(k, r) : make_float2(r, k); }
};

// a pair of floats at an even index, one load
__device__ __forceinline__ float2 load2(const float* __restrict__ v, int32_t o) { return *(const float2*)(v + o); }
__device__ __forceinline__ void   store2(float* __restrict__ v, int32_t o, float2 x) { *(float2*)(v + o) = x; }

// where a pair's neighbours lie, for brick s with the neighbour slots nb[0..5]: o the pair, xm and xp the
// cells before and after it, ym .. zp the adjacent pairs (o where there is no neighbour), h: which there are
struct PairNeighbours {
    int32_t o, xm, xp, ym, yp, zm, zp;
    bool    hxm, hxp, hym, hyp, hzm, hzp;
    __device__ __forceinline__ PairNeighbours(const int32_t* __restrict__ nb, int32_t s, const BrickPair& c) {
        const int l = c.even;
        o   = s * 512 + l;
        hxm = c.px > 0 || nb[0] >= 0;
        hxp = c.px < 3 || nb[1] >= 0;
        hym = c.ly > 0 || nb[2] >= 0;
        hyp = c.ly < 7 || nb[3] >= 0;
        hzm = c.lz > 0 || nb[4] >= 0;
        hzp = c.lz < 7 || nb[5] >= 0;
        xm  = c.px > 0 ? o - 1 : (hxm ? nb[0] * 512 + l + 7 : o);
        xp  = c.px < 3 ? o + 2 : (hxp ? nb[1] * 512 + l - 6 : o);
        ym  = c.ly > 0 ? o - 8 : (hym ? nb[2] * 512 + l + 56 : o);
        yp  = c.ly < 7 ? o + 8 : (hyp ? nb[3] * 512 + l - 56 : o);
        zm  = c.lz > 0 ? o - 64 : (hzm ? nb[4] * 512 + l + 448 : o);
        zp  = c.lz < 7 ? o + 64 : (hzp ? nb[5] * 512 + l - 448 : o);
    }
};

// a pair's couplings: cx, cy, cz its own (upwards), xm, ym, zm those of its lower neighbours
struct PairCoupling {
    float2 cx, cy, cz, ym, zm;
    float  xm;
};
template<class L> __device__ __forceinline__ PairCoupling pair_coupling(const L& A, const PairNeighbours& n, bool uni) {
    const float  c = A.uni.c;
    const float2 c2 = make_float2(c, c);
    PairCoupling w{c2, c2, c2, c2, c2, c};
    if(!uni) {
        w.cx = load2(A.cx, n.o);
        w.cy = load2(A.cy, n.o);
        w.cz = load2(A.cz, n.o);
        w.ym = load2(A.cy, n.ym);
        w.zm = load2(A.cz, n.zm);
        w.xm = A.cx[n.xm];
    }
    return w;
}

// A cell's row of A in the brick smoothers, divided by the diagonal and with the sign of the update
// x = b/d - sum (a/d) x (a coupling to a missing neighbour is 0 and that neighbour's halo entry holds 0, so
// all six terms are added unconditionally). The coupling inside the pair (`in`) takes the other cell's value
// from a register. Five LDS reads and seven multiply-adds in two chains, against six reads and fourteen
// operations in one: the half-sweeps are a serial chain.
struct SmoothRow {
    float zm, ym, out, in, yp, zp, bs;
    // the cell's new value, x at its tile entry; pair: the other cell of its pair
    __device__ __forceinline__ float solved(const float* x, int off, float pair) const {
        const float p = __builtin_fmaf(out, x[off], __builtin_fmaf(ym, x[-kTileRow], __builtin_fmaf(zm, x[-kTilePlane], bs)));
        return p + __builtin_fmaf(zp, x[kTilePlane], __builtin_fmaf(yp, x[kTileRow], in * pair));
    }
};
// the rows of the pair's red and black cell (bs left 0)
__device__ __forceinline__ void smooth_rows(const PairCoupling& w, float2 inv, const PairNeighbours& n, const BrickPair& c, SmoothRow& R, SmoothRow& K) {
    const SmoothRow E{n.hzm ? -w.zm.x * inv.x : 0.f, n.hym ? -w.ym.x * inv.x : 0.f, n.hxm ? -w.xm * inv.x : 0.f, -w.cx.x * inv.x,
                      n.hyp ? -w.cy.x * inv.x : 0.f, n.hzp ? -w.cz.x * inv.x : 0.f, 0.f};
    const SmoothRow O{n.hzm ? -w.zm.y * inv.y : 0.f, n.hym ? -w.ym.y * inv.y : 0.f, n.hxp ? -w.cx.y * inv.y : 0.f, -w.cx.x * inv.y,
                      n.hyp ? -w.cy.y * inv.y : 0.f, n.hzp ? -w.cz.y * inv.y : 0.f, 0.f};
    R = c.swap ? O : E;
    K = c.swap ? E : O;
}

// xpre + omega * x_coarse(parent) for an unknown, xpre otherwise (x + omega P x_c); xc: the coarse value,
// any where the parent brick is missing (has: it is there)
__device__ __forceinline__ float mg_prolonged(float xpre, float xc, bool has, float inv, float omega) {
    return has && inv != 0.f ? xpre + omega * xc : xpre;
}

// the brick's one-cell halo (6 faces x 64 cells) in LDS: the neighbouring bricks' corrected values, 0 where
// there is none. A wave a face, so the face and its neighbour are scalars. The parent of the neighbour brick
// is this brick's parent, or that one's neighbour across the face when this brick is on the parent's face.
__device__ __forceinline__ void smooth_halo(const LevelDev& L, const LevelDev& C, float omega, int s, float* xs) {
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), a = threadIdx.x & 7, e = threadIdx.x >> 3 & 7;
#pragma unroll
    for(int q = 0; q < 2; ++q) {
        const int d = w + 4 * q;
        if(d >= 6) break;
        const int32_t n  = L.nbr[6 * s + d];
        const int     sa = d < 2 ? kTileRow : 1, se = d < 4 ? kTilePlane : kTileRow, sd = d < 2 ? 1 : (d < 4 ? kTileRow : kTilePlane);
        float         v  = 0.f;
        if(n >= 0) {
            // the cell's coordinates in the neighbour: m across the face, a and e along it
            const int     m = d & 1 ? 0 : 7, lx = d < 2 ? m : a, ly = d < 2 ? a : (d < 4 ? m : e), lz = d < 4 ? e : m;
            const int32_t o = n * 512 + (lz * 8 + ly) * 8 + lx;
            const int     own = L.ptab[8 * s + 7], odd = own ^ 1 << (d >> 1);  // parities of the brick's, the neighbour's coordinates
            const bool    cross = (own >> (d >> 1) & 1) == (d & 1);
            const int32_t cs = L.ptab[8 * s + (cross ? d : 6)];
            const int     cl = (((odd >> 2 & 1) * 4 + lz / 2) * 8 + (odd >> 1 & 1) * 4 + ly / 2) * 8 + (odd & 1) * 4 + lx / 2;
            v                = mg_prolonged(L.r[o], C.x[cs < 0 ? 0 : cs * 512 + cl], cs >= 0, L.invdiag[o], omega);
        }
        xs[(1 + a) * sa + (1 + e) * se + (d & 1 ? 9 : 0) * sd] = v;
    }
}

// Brick-hybrid Gauss-Seidel: one block per brick runs `sweeps` red-black sweeps (pre-smoother) or
// black-red sweeps (post-smoother) on its 512 cells in LDS, with the x of neighbouring bricks held at
// their values on entry (Jacobi between bricks). For the brick's own system A_BB the red-black and
// black-red sequences are transposes of each other, so the pre- and post-smoothers are adjoint and
// the V-cycle stays symmetric. Pre-smoother: starts from x = 0 (every V-cycle does) and writes L.r.
// Post-smoother (kPost): starts from the coarse-grid-corrected L.r + omega * P x_coarse, formed here for
// the brick and its halo, and writes L.x. (On the finest level the correction was once a streaming pass of
// its own, 12.9 us at 9593 bricks and a launch; with the parents from the brick tables it costs the smoother
// 10: 33.7 -> 43.8 us, at 1309 bricks 7.7 -> 9.2 for a pass of 3.5.) Input and output are different arrays, so no block reads what another writes. Each of the 256 threads owns
// an x-adjacent pair of cells, one of each colour, so every thread updates one cell per half-sweep.
// kDot (finest level, post-smoother): also writes the brick's partial of z.r (z = the result,
// r = L.b) to pz[slot], the PCG's next rho.
template<bool kPost, bool kDot>
__device__ __forceinline__ void mg_smooth_one(const LevelDev& L, const LevelDev& C, float omega, int sweeps, double* __restrict__ pz, int s,
                                              const BrickPair& c, float2 b, float* xs, double* sh) {
    const int            t = threadIdx.x;
    const PairNeighbours n(L.nbr + 6 * s, s, c);
    const bool           uni = L.uni.is(s);
    const PairCoupling   w   = pair_coupling(L, n, uni);
    const float2         inv = uni ? make_float2(L.uni.inv, L.uni.inv) : load2(L.invdiag, n.o);
    float                zr, zb;
    SmoothRow            R, K;
    if(kPost) {
        const int32_t cs = L.ptab[8 * s + 6];
        const float   xc = C.x[cs < 0 ? 0 : cs * 512 + c.parent(L.ptab[8 * s + 7])];
        float2        xv = load2(L.r, n.o);
        xv = make_float2(mg_prolonged(xv.x, xc, cs >= 0, inv.x, omega), mg_prolonged(xv.y, xc, cs >= 0, inv.y, omega));
        smooth_halo(L, C, omega, s, xs);
        xs[c.cr] = zr = c.red(xv);
        xs[c.cb] = zb = c.black(xv);
    } else {  // x = 0, and 0 around it
        for(int e = t; e < kTile / 4; e += 256) ((float4*)xs)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
    }
    smooth_rows(w, inv, n, c, R, K);
    R.bs = c.red(b) * c.red(inv);
    K.bs = c.black(b) * c.black(inv);
    if(!kPost) {
        xs[c.cr] = zr = R.bs;  // the first red half-sweep
        zb            = 0.f;
    }
    auto red   = [&] { xs[c.cr] = zr = R.solved(xs + c.cr, c.offR, zb); };
    auto black = [&] { xs[c.cb] = zb = K.solved(xs + c.cb, -c.offR, zr); };
    __syncthreads();
    for(int it = 0; it < sweeps; ++it) {
        if(kPost) black();
        else if(it) red();
        if(kPost || it) __syncthreads();
        if(kPost) red();
        else black();
        __syncthreads();
    }
    store2(kPost ? L.x : L.r, n.o, c.cells(zr, zb));
    if(kDot) {
        const double d = block_sum<256>((double)zr * (double)c.red(b) + (double)zb * (double)c.black(b), sh);
        if(t == 0) pz[s] = d;
    }
    __syncthreads();  // xs is reused by the workgroup's next brick
}

template<bool kPost, bool kDot>
struct k_mg_smooth_brick {
    static constexpr int kThreads = 256;
    LevelDev L;
    LevelDev C;
    float omega;
    int sweeps;
    const PcgState* __restrict__ st;
    double* __restrict__ pz;
    __device__ void operator()(Blk blk) const {
        __shared__ __align__(16) float xs[kTile];  // the brick and a one-cell halo
        __shared__ double sh[4];
        if(st && st->done) return;
        const BrickPair c(threadIdx.x);
        for(uint32_t v = blk.id; v < L.nSlots; v += blk.n) {
            const int s = (int)xcd_slot(v, L.nSlots);
            mg_smooth_one<kPost, kDot>(L, C, omega, sweeps, pz, s, c, load2(L.b, s * 512 + c.even), xs, sh);
        }
    }
};

// The PCG update fused with the V-cycle's first step on the finest level (multigrid): per brick,
// x += alpha s and r -= alpha q (PCGSolver.cpp:178-181), the brick's max|r| to the max words, then the
// pre-smoother on b = r, which reads only the brick's own cells (it starts from x = 0). The finest
// level's r array is the PCG's q buffer: this brick's q is read before the smoother overwrites it.
// Per cell the same arithmetic as k_pcg_update followed by k_mg_smooth_brick<false, false>.
// kFold (small systems): alpha (k_pcg_alpha) is formed here from nPart <= kFoldMax partials of s.q.
template<bool kFold>
struct k_pcg_update_pre {
    static constexpr int kThreads = 256;
    const float* __restrict__ s;
    float* __restrict__ x;
    LevelDev L;  // the finest level: L.b = r, L.r = q
    float omega;
    int sweeps;
    PcgState* st;
    uint32_t* maxWords;
    const double* __restrict__ sq;
    int nPart;
    __device__ void operator()(Blk blk) const {
        __shared__ __align__(16) float xs[kTile];
        __shared__ double sh[kFoldMax / 64];
        const int  t     = threadIdx.x;
        const bool done  = st->done != 0;
        float      alpha = 0.f;
        double     A = 0, al = 0;
        if(kFold) {
            // The first workgroup records alpha in the state, at the end (see k_mg_residual_restrict), or the
            // stop when the sum ends the solve. That store may fall between the reads of the flag by two waves
            // of another workgroup, so every wave takes part in the fold, whatever it read, and leaves by the
            // sum: one that saw the stop of this launch has the same sum in front of it as one that did not.
            // (Leaving before it, a wave would miss its part of the fold.) A stop of an earlier launch is seen by all.
            A  = fold_all<256>(sq, nPart, sh);
            al = st->rho / A;
            if(done) return;
            if(A < (double)kFltMin) {
                if(blk.id == 0 && t == 0) {
                    st->tmp     = A;
                    st->done    = 1;
                    st->success = 1;
                    st->iter += 1;
                }
                return;
            }
            alpha = (float)al;
        } else {
            if(done) return;
            alpha = (float)st->alpha;
        }
        const BrickPair c(t);
        for(uint32_t v = blk.id; v < L.nSlots; v += blk.n) {
            const int     slot = (int)xcd_slot(v, L.nSlots);
            const int32_t o    = slot * 512 + c.even;
            const float2  sv = load2(s, o), qv = load2(L.r, o);
            float2        xv = load2(x, o), rv = load2(L.b, o);
            xv = make_float2(xv.x + alpha * sv.x, xv.y + alpha * sv.y);
            rv = make_float2(rv.x + (-alpha) * qv.x, rv.y + (-alpha) * qv.y);
            store2(x, o, xv);
            store2(L.b, o, rv);
            const double m = block_max<256>(fmax((double)fabsf(rv.x), (double)fabsf(rv.y)), sh);
            mg_smooth_one<false, false>(L, L, omega, sweeps, nullptr, slot, c, rv, xs, sh);
            if(t == 0) max_words_put(maxWords, v, (float)m);
        }
        if(kFold && blk.id == 0 && t == 0) {
            st->tmp   = A;
            st->alpha = al;
        }
    }
};

// r = b - A x on level F with the pre-smoothed x (held in F.r), summed over each 2x2x2 group into
// the coarse right-hand side (P^T r). A group's eight cells lie in one fine brick, so the block of a
// fine brick writes the 64 coarse cells it covers; r itself is never stored. Coarse cells without an
// active child brick keep the zeros they get when the hierarchy is built. A thread's pair of cells and its
// partners in the group, lanes ^ 4 and ^ 32, form the sum.
// kStop (finest level, after a fused update): first the iteration's stop test, on the max words; the first
// workgroup records it. A wave of another workgroup that sees the stop it records leaves early, which is no
// matter: the V-cycle ends with this iteration, and no wave here waits for another. It records it at the end:
// after a store to the state the compiler loads the tables, which may overlap it for all it knows, by vector
// instructions (the restriction of 9593 bricks 13.7 -> 30 us).
// At most kMaxRedBlocks workgroups take the bricks in turn then, for the words' read before the first: 19.8 us
// at 9593 bricks against 22.8 with a workgroup a brick.
template<bool kStop>
struct k_mg_residual_restrict {
    static constexpr int kThreads = 256;
    LevelDev F;
    LevelDev C;
    PcgState* st;
    const uint32_t* maxWords;
    __device__ void operator()(Blk blk) const {
        const int t = threadIdx.x;
        float     B = 0.f;
        if(kStop) {
            const float    w = __uint_as_float(maxWords[kMaxWordStep * (t & 63)]), tol = st->tol;
            const uint32_t done = st->done;
            if(done) return;
            B = wave_max(w);
            if(B < tol) {
                if(blk.id == 0 && t == 0) pcg_stop_test(*st, B);
                return;
            }
        } else if(st && st->done) {
            return;
        }
        const BrickPair c(t);
        for(uint32_t v = blk.id; v < F.nSlots; v += blk.n) {
            const int            s = (int)xcd_slot(v, F.nSlots);
            const PairNeighbours n(F.nbr + 6 * s, s, c);
            const bool           uni = F.uni.is(s);
            const PairCoupling   w   = pair_coupling(F, n, uni);
            const float2         dia = uni ? make_float2(F.uni.d, F.uni.d) : load2(F.diag, n.o);
            const float2         b = load2(F.b, n.o), x = load2(F.r, n.o), ym = load2(F.r, n.ym), yp = load2(F.r, n.yp), zm = load2(F.r, n.zm),
                         zp = load2(F.r, n.zp);
            const float xm = F.r[n.xm], xp = F.r[n.xp];
            // a missing neighbour adds its zero coupling times the pair's own x
            auto offdiag = [&](float czm, float vzm, float cym, float vym, float cxm, float vxm, float cxp, float vxp, float cyp, float vyp, float czp, float vzp) {
                float acc = 0.f;
                acc += (n.hzm ? czm : 0.f) * vzm;
                acc += (n.hym ? cym : 0.f) * vym;
                acc += cxm * vxm;
                acc += cxp * vxp;
                acc += (n.hyp ? cyp : 0.f) * vyp;
                acc += (n.hzp ? czp : 0.f) * vzp;
                return acc;
            };
            const float r0 = b.x - (dia.x * x.x + offdiag(w.zm.x, zm.x, w.ym.x, ym.x, n.hxm ? w.xm : 0.f, xm, w.cx.x, x.y, w.cy.x, yp.x, w.cz.x, zp.x));
            const float r1 = b.y - (dia.y * x.y + offdiag(w.zm.y, zm.y, w.ym.y, ym.y, w.cx.x, x.x, n.hxp ? w.cx.y : 0.f, xp, w.cy.y, yp.y, w.cz.y, zp.y));
            // the odd y of the 2x2x2 group lies in lane ^ 4, the odd z in lane ^ 32
            const float   e = r0 + r1, ey = e + __shfl_xor(e, 4), sum = ey + __shfl_xor(ey, 32);
            const int32_t cs = F.ptab[8 * s + 6];
            if(!(c.ly & 1) && !(c.lz & 1) && cs >= 0) C.b[cs * 512 + c.parent(F.ptab[8 * s + 7])] = sum;
        }
        if(kStop && blk.id == 0 && t == 0) pcg_stop_test(*st, B);
    }
};

// A coarsest level of more than one brick, which only an axis of more than 8 * 2^15 cells leaves (the last of
// kMaxMgLevels levels; k_mg_tail solves one brick): x = 0, then `sweeps` red-black sweeps followed by `sweeps`
// black-red sweeps (symmetric), all inside one block
struct k_mg_coarsest {
    static constexpr int kThreads = 1024;
    LevelDev L;
    int sweeps;
    const PcgState* __restrict__ st;
    __device__ void operator()(Blk blk) const {
        if(st && st->done) return;
        const uint32_t n = L.nSlots * 512;
        for(uint32_t t = threadIdx.x; t < n; t += blockDim.x) L.x[t] = 0.f;
        __syncthreads();
        for(int it = 0; it < 2 * sweeps; ++it) {
            for(int half = 0; half < 2; ++half) {
                const int color = (it < sweeps) ? half : 1 - half;
                for(uint32_t t = threadIdx.x; t < n; t += blockDim.x) {
                    const int s = (int)(t >> 9), l = (int)(t & 511);
                    if(cell_color(L, s, l) != color) continue;
                    L.x[t] = (L.b[t] - level_offdiag_sum(L, s, l, L.x)) * L.invdiag[t];
                }
                __syncthreads();
            }
        }
    }
};

//==================================================================================================
// The reference's preconditioner: natural-order incomplete Cholesky IC(0) with the 0.25 pivot
// safeguard (PCGSolver.cpp:398-466, minDiagonalRatio PCGSolver.h:88-89) and its two triangular
// solves (PCGSolver.cpp:243-269), level-scheduled over the hyperplanes i + j + k = h. On the 7-point
// stencil every lower neighbour of a cell (-x, -y, -z) lies on plane h - 1 and every upper neighbour
// on h + 1, so one launch per plane, in plane order, reproduces the sequential recurrences; each
// cell applies its neighbours' terms in the reference's order (by ascending natural index: -z, -y,
// -x going forward; +x, +y, +z coming back), with the same FP32 roundings. 3n - 2 dependent launches
// per sweep: latency-bound, used to compare iterates with the reference's preconditioner, not for
// speed. Cells outside the system (solid, air, the outer layer) have a zero diagonal and a zero
// factor, so they contribute nothing and get z = 0.
//==================================================================================================
struct Ic0Dev {
    const int32_t* brickSlot;
    const float *  diag, *cx, *cy, *cz;  // A: diagonal and the couplings to +x, +y, +z
    float *        inv, *lx, *ly, *lz;   // 1/sqrt(pivot); L entries below the diagonal (column-scaled)
};

__device__ __forceinline__ int32_t sys_cell(const int32_t* __restrict__ brickSlot, const GridGeom& g, int i, int j, int k) {
    if(i < 0 || j < 0 || k < 0) return -1;
    const int32_t s = brickSlot[((k >> 3) * g.nby + (j >> 3)) * g.nbx + (i >> 3)];
    return s < 0 ? -1 : s * 512 + ((k & 7) * 8 + (j & 7)) * 8 + (i & 7);
}

// the cell (i, j, k = h - i - j) of plane h owned by this thread, or -1
__device__ __forceinline__ int32_t ic0_plane_cell(Blk blk, const Ic0Dev& D, const GridGeom& g, int h, int& i, int& j, int& k) {
    const uint32_t t = blk.id * blockDim.x + threadIdx.x;
    if(t >= (uint32_t)g.nx * (uint32_t)g.ny) return -1;
    i = (int)(t % (uint32_t)g.nx);
    j = (int)(t / (uint32_t)g.nx);
    k = h - i - j;
    if(k < 0 || k >= g.nz) return -1;
    return sys_cell(D.brickSlot, g, i, j, k);
}

// pivot d = a_oo - L(o,-z)^2 - L(o,-y)^2 - L(o,-x)^2 (the column updates of the lower neighbours,
// in their processing order), inv = 1/sqrt(d), or 1/sqrt(a_oo) when d < 0.25 a_oo; then the column
// below the diagonal is scaled: L(+x,o) = a(o,+x) * inv, and likewise +y, +z
struct k_ic0_factor_plane {
    static constexpr int kThreads = kBlock;
    Ic0Dev D;
    GridGeom g;
    int h;
    __device__ void operator()(Blk blk) const {
    #pragma clang fp contract(off)
        int           i, j, k;
        const int32_t o = ic0_plane_cell(blk, D, g, h, i, j, k);
        if(o < 0) return;
        const float a = D.diag[o];
        float       inv;
        if(a < kFltMin) {
            inv = a;  // row skipped by the factorisation (PCGSolver.cpp:419-421): its couplings are zero
        } else {
            const int32_t mz = sys_cell(D.brickSlot, g, i, j, k - 1), my = sys_cell(D.brickSlot, g, i, j - 1, k),
                          mx = sys_cell(D.brickSlot, g, i - 1, j, k);
            float d = a;
            if(mz >= 0) {
                const float l = D.lz[mz];
                d -= l * l;
            }
            if(my >= 0) {
                const float l = D.ly[my];
                d -= l * l;
            }
            if(mx >= 0) {
                const float l = D.lx[mx];
                d -= l * l;
            }
            inv = d < 0.25f * a ? 1.0f / sqrtf(a) : 1.0f / sqrtf(d);
        }
        D.inv[o] = inv;
        const bool skipped = a < kFltMin;  // an unscaled zero column
        D.lx[o]  = skipped ? D.cx[o] : D.cx[o] * inv;
        D.ly[o]  = skipped ? D.cy[o] : D.cy[o] * inv;
        D.lz[o]  = skipped ? D.cz[o] : D.cz[o] * inv;
    }
};

// forward solve, plane h: y_o = (((r_o - L(o,-z) y_-z) - L(o,-y) y_-y) - L(o,-x) y_-x) * inv_o
struct k_ic0_lower_plane {
    static constexpr int kThreads = kBlock;
    Ic0Dev D;
    GridGeom g;
    int h;
    const float* __restrict__ r;
    float* __restrict__ y;
    const PcgState* __restrict__ st;
    __device__ void operator()(Blk blk) const {
    #pragma clang fp contract(off)
        if(st && st->done) return;
        int           i, j, k;
        const int32_t o = ic0_plane_cell(blk, D, g, h, i, j, k);
        if(o < 0) return;
        const int32_t mz = sys_cell(D.brickSlot, g, i, j, k - 1), my = sys_cell(D.brickSlot, g, i, j - 1, k),
                      mx = sys_cell(D.brickSlot, g, i - 1, j, k);
        float v = r[o];
        if(mz >= 0) v -= D.lz[mz] * y[mz];
        if(my >= 0) v -= D.ly[my] * y[my];
        if(mx >= 0) v -= D.lx[mx] * y[mx];
        y[o] = v * D.inv[o];
    }
};

// backward solve in place, plane h (descending): z_o = (((y_o - L(+x,o) z_+x) - L(+y,o) z_+y) -
// L(+z,o) z_+z) * inv_o
struct k_ic0_upper_plane {
    static constexpr int kThreads = kBlock;
    Ic0Dev D;
    GridGeom g;
    int h;
    float* __restrict__ z;
    const PcgState* __restrict__ st;
    __device__ void operator()(Blk blk) const {
    #pragma clang fp contract(off)
        if(st && st->done) return;
        int           i, j, k;
        const int32_t o = ic0_plane_cell(blk, D, g, h, i, j, k);
        if(o < 0) return;
        const int32_t px = i + 1 < g.nx ? sys_cell(D.brickSlot, g, i + 1, j, k) : -1;
        const int32_t py = j + 1 < g.ny ? sys_cell(D.brickSlot, g, i, j + 1, k) : -1;
        const int32_t pz = k + 1 < g.nz ? sys_cell(D.brickSlot, g, i, j, k + 1) : -1;
        float         v  = z[o];
        if(px >= 0) v -= D.lx[o] * z[px];
        if(py >= 0) v -= D.ly[o] * z[py];
        if(pz >= 0) v -= D.lz[o] * z[pz];
        z[o] = v * D.inv[o];
    }
};

// partial z.r for the PCG (after the preconditioner wrote z)
struct k_pcg_dot_zr {
    static constexpr int kThreads = 512;
    const float* __restrict__ z;
    const float* __restrict__ r;
    uint32_t nSlots;
    const PcgState* __restrict__ st;
    double* __restrict__ pa;
    __device__ void operator()(Blk blk) const {
        __shared__ double sh[8];
        if(st && st->done) return;
        double d = 0;
        for(uint32_t slot = blk.id; slot < nSlots; slot += blk.n) {
            const size_t o = (size_t)slot * 512 + threadIdx.x;
            d += (double)z[o] * (double)r[o];
        }
        d = block_sum<512>(d, sh);
        if(threadIdx.x == 0) pa[blk.id] = d;
    }
};

}  // namespace bnn

namespace bnn {

// The V-cycle's smallest levels in one launch. On levels of a few bricks every kernel of the cycle costs
// its own dependent loads and its launch (5-7 us each, three a level, 11 for a coarsest solve by one
// wavefront), whatever its work. Here one workgroup takes the levels lv[0] (at most 8 bricks) to the
// coarsest (one brick): all their x tiles (a brick and its one-cell halo) stay in LDS, a right-hand side
// goes to the next level through that level's tile, and the coefficients of the first two levels and the
// coarsest are loaded once, at the start. Four groups of 256 threads own a brick each (on lv[0] up to two in turn;
// thread = an x-adjacent pair of cells, one of each colour). The steps are those of k_mg_smooth_brick and
// k_mg_residual_restrict; coarsest level: x = 0, `coarsest` red-black and as many black-red sweeps. Input
// lv[0].b, output lv[0].x. The first red half-sweep from x = 0 and the black one that would repeat the one
// before it are left out. Bound by what four waves a SIMD issue (16 cycles an instruction on lv[0]) and by
// the chain of half-sweeps (260 cycles each on the coarsest level): so pairs of coefficients are loaded as
// one, tables and own coefficients before anything waits, a halo's face and neighbour are scalars. 13 us
// for two levels, 20 for three (16 and 25 before that and the tile's strides), against 27 and 42 in
// separate kernels plus 4 or 7 launches.
struct k_mg_tail {
    static constexpr int kThreads = 1024;
    static constexpr int kLevels = 5, kTop = 8, kRest = 4, kTiles = 16;  // levels; bricks on lv[0], on each other level, in all
    LevelDev lv[kLevels];
    int      nLev;
    float    omega;
    int      sweeps, coarsest;
    const PcgState* __restrict__ st;

    // a cell's row of A and its diagonal
    struct Row : SmoothRow {
        float diag;
        __device__ __forceinline__ void rhs(float b) { bs = diag > 0.f ? b / diag : 0.f; }
    };
    static __device__ __forceinline__ int tile_at(int l) { return tile_index(l & 7, (l >> 3) & 7, l >> 6); }
    // what a pair's rows take besides its lower neighbours' couplings
    struct Own {
        float2 diag, inv, cx, cy, cz;
    };
    static __device__ __forceinline__ Own own(const LevelDev& L, int32_t o) {
        return Own{load2(L.diag, o), load2(L.invdiag, o), load2(L.cx, o), load2(L.cy, o), load2(L.cz, o)};
    }
    // the rows of the pair's red and black cell; nb: the brick's six neighbour slots
    static __device__ __forceinline__ void rows(const LevelDev& L, const int32_t* nb, const Own& w, int32_t s, const BrickPair& c, Row& R, Row& K) {
        const PairNeighbours n(nb, s, c);
        smooth_rows(PairCoupling{w.cx, w.cy, w.cz, load2(L.cy, n.ym), load2(L.cz, n.zm), L.cx[n.xm]}, w.inv, n, c, R, K);
        R.diag = c.red(w.diag);
        K.diag = c.black(w.diag);
    }
    // one half-sweep over the group's n bricks (4 tiles apart): cells of one colour read only the other.
    // own: the cells' values, pair: those of the other colour
    template<int kTurns> static __device__ __forceinline__ void half(const Row* R, float* x, int off, float* own, const float* pair, int n) {
#pragma unroll
        for(int q = 0; q < kTurns; ++q)
            if(q < n) own[q] = R[q].solved(x + 4 * kTile * q, off, pair[q]);
#pragma unroll
        for(int q = 0; q < kTurns; ++q)
            if(q < n) x[4 * kTile * q] = own[q];
    }
    // the first red half-sweep, from x = 0
    template<int kTurns> static __device__ __forceinline__ void first(const Row* R, float* x, float* own, int n) {
#pragma unroll
        for(int q = 0; q < kTurns; ++q)
            if(q < n) x[4 * kTile * q] = own[q] = R[q].bs;
    }
    // the tiles' halos from the neighbouring bricks (where there is none they stay 0): a wave a face, so the
    // face and its neighbour are scalars
    static __device__ __forceinline__ void halos(float* xs, const int32_t (*nb)[8], int S) {
        constexpr int kWaves = kThreads / 64, kFaces = 6 * kTop / kWaves;
        const int     w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), a = threadIdx.x & 7, e = threadIdx.x >> 3 & 7;
        int32_t       n[kFaces];
#pragma unroll
        for(int q = 0; q < kFaces; ++q) {
            const int f = w + kWaves * q;
            n[q]        = f < 6 * S ? nb[f / 6][f % 6] : -1;
        }
#pragma unroll
        for(int q = 0; q < kFaces; ++q) {
            const int f = w + kWaves * q, s = f / 6, d = f % 6, m = __builtin_amdgcn_readfirstlane(n[q]);
            if(m < 0) continue;
            // along the face's two axes; across it the halo entry and, step further, the cell it mirrors
            const int sa = d < 2 ? kTileRow : 1, se = d < 4 ? kTilePlane : kTileRow, sd = d < 2 ? 1 : (d < 4 ? kTileRow : kTilePlane);
            const int to = (1 + a) * sa + (1 + e) * se + (d & 1 ? 9 : 0) * sd;
            xs[kTile * s + to] = xs[kTile * m + (d & 1 ? -8 : 8) * sd + to];
        }
    }
    // pre-smoother from x = 0 on the level's tiles, then the residual's 2x2x2 sums to the next level's tiles
    // (its right-hand side) and to its b (for the way up)
    template<int kTurns>
    __device__ __forceinline__ void down(const Row* R, const Row* K, const BrickPair& c, float* xs, const int32_t (*nb)[8], int S, int grp, const LevelDev& C) const {
        const int n = (S - grp + 3) >> 2;  // bricks grp, grp + 4, ..
        float*    x = xs + kTile * grp;
        float     vr[kTurns] = {}, vb[kTurns] = {};
        first<kTurns>(R, x + c.cr, vr, n);
        __syncthreads();
        for(int it = 0; it < sweeps; ++it) {
            if(it) {
                half<kTurns>(R, x + c.cr, c.offR, vr, vb, n);
                __syncthreads();
            }
            half<kTurns>(K, x + c.cb, -c.offR, vb, vr, n);
            __syncthreads();
        }
        halos(xs, nb, S);
        __syncthreads();
#pragma unroll
        for(int q = 0; q < kTurns; ++q)
            if(q < n) {
                const float* y  = x + 4 * kTile * q;
                const float  rr = R[q].diag * (R[q].solved(y + c.cr, c.offR, vb[q]) - vr[q]);
                const float  rk = K[q].diag * (K[q].solved(y + c.cb, -c.offR, vr[q]) - vb[q]);
                // the x pair is this thread's, the odd y lies in lane ^ 4, the odd z in lane ^ 32
                const float e = rr + rk, ey = e + __shfl_xor(e, 4), sum = ey + __shfl_xor(ey, 32);
                const int   par = nb[grp + 4 * q][6];
                if(!(c.ly & 1) && !(c.lz & 1) && par >= 0) {
                    const int   cl  = c.parent(nb[grp + 4 * q][7]);
                    xs[kTile * (S + par) + tile_at(cl)] = sum;
                    C.b[par * 512 + cl]                = sum;
                }
            }
        __syncthreads();
    }
    // coarse-grid correction, then the post-smoother
    template<int kTurns>
    __device__ __forceinline__ void up(const Row* R, const Row* K, const BrickPair& c, float* xs, const int32_t (*nb)[8], int S, int grp) const {
        const int n = (S - grp + 3) >> 2;
        float*    x = xs + kTile * grp;
        float     vr[kTurns] = {}, vb[kTurns] = {};
#pragma unroll
        for(int q = 0; q < kTurns; ++q)
            if(q < n) {
                const int par = nb[grp + 4 * q][6];
                float*    y   = x + 4 * kTile * q;
                vr[q]         = y[c.cr];
                vb[q]         = y[c.cb];
                if(par >= 0) {
                    const float xc = xs[kTile * (S + par) + tile_at(c.parent(nb[grp + 4 * q][7]))];
                    if(R[q].diag > 0.f) y[c.cr] = vr[q] = vr[q] + omega * xc;
                    if(K[q].diag > 0.f) y[c.cb] = vb[q] = vb[q] + omega * xc;
                }
            }
        __syncthreads();
        halos(xs, nb, S);
        __syncthreads();
        for(int it = 0; it < sweeps; ++it) {
            half<kTurns>(K, x + c.cb, -c.offR, vb, vr, n);
            __syncthreads();
            half<kTurns>(R, x + c.cr, c.offR, vr, vb, n);
            __syncthreads();
        }
    }
    __device__ void operator()(Blk) const {
        __shared__ __align__(16) float xs[kTiles * kTile];
        __shared__ int32_t nb[kTiles][8];  // per brick: six neighbour slots, parent slot, parities of its coordinates
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));  // keeps the batched form's loop over scenes from holding the lane's constants in registers
        const int       grp = t >> 8;
        const BrickPair c(t & 255);
        // the brick tables and the pairs' own coefficients of the first two levels and the coarsest, before
        // anything waits: the lower neighbours' follow when the tables are in LDS
        int32_t tab[kLevels];
#pragma unroll
        for(int l = 0; l < kLevels; ++l) {
            const int s = t >> 3, d = t & 7;
            tab[l] = -1;
            if(l < nLev && s < (int)lv[l].nSlots) {
                if(d < 6) tab[l] = lv[l].nbr[6 * s + d];
                else if(l + 1 < nLev) tab[l] = lv[l].ptab[8 * s + d];
            }
        }
        const int last = nLev - 1;
        const int S0   = nLev > 1 ? (int)lv[0].nSlots : 0;
        Own       own0[2], own1, ownC;
        float2    b0[2];
#pragma unroll
        for(int q = 0; q < 2; ++q)
            if(grp + 4 * q < S0) {
                own0[q] = own(lv[0], (grp + 4 * q) * 512 + c.even);
                b0[q]   = load2(lv[0].b, (grp + 4 * q) * 512 + c.even);
            }
        if(nLev > 2 && grp < (int)lv[1].nSlots) own1 = own(lv[1], grp * 512 + c.even);
        if(grp == 0) ownC = own(lv[last], c.even);
        if(st && st->done) return;
        int base = 0;
#pragma unroll
        for(int l = 0; l < kLevels; ++l)
            if(l < nLev) {
                const int S = (int)lv[l].nSlots;
                if(t < 8 * S) nb[base + (t >> 3)][t & 7] = tab[l];
                base += S;
            }
        for(int e = t; e < base * (kTile / 4); e += kThreads) ((float4*)xs)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
        Row R0[2], K0[2], R1[1], K1[1], RC, KC;  // the first level, the second (or a later one), the coarsest
#pragma unroll
        for(int q = 0; q < 2; ++q) {
            const int s = grp + 4 * q;
            if(s < S0) {
                rows(lv[0], nb[s], own0[q], s, c, R0[q], K0[q]);
                R0[q].rhs(c.red(b0[q]));
                K0[q].rhs(c.black(b0[q]));
            }
        }
        const int lastAt = base - 1;  // the coarsest level's only tile
        if(nLev > 2 && grp < (int)lv[1].nSlots) rows(lv[1], nb[S0 + grp], own1, grp, c, R1[0], K1[0]);
        if(grp == 0) rows(lv[last], nb[lastAt], ownC, 0, c, RC, KC);
        // a later level's rows, when it is its turn
        auto later = [&](int l, int at) {
            if(grp < (int)lv[l].nSlots) rows(lv[l], nb[at + grp], own(lv[l], grp * 512 + c.even), grp, c, R1[0], K1[0]);
        };
        // the right-hand side that the finer level left in the tile; x starts from 0
        auto take = [&](Row& R, Row& K, int at) {
            float* x = xs + kTile * at;
            R.rhs(x[c.cr]);
            K.rhs(x[c.cb]);
            x[c.cr] = x[c.cb] = 0.f;
        };
        if(nLev > 1) down<2>(R0, K0, c, xs, nb, S0, grp, lv[1]);
        base = S0;
        for(int l = 1; l < last; ++l) {
            const int S = (int)lv[l].nSlots;
            if(l > 1) later(l, base);
            if(grp < S) take(R1[0], K1[0], base + grp);
            down<1>(R1, K1, c, xs + kTile * base, nb + base, S, grp, lv[l + 1]);
            base += S;
        }
        {  // coarsest level, one brick
            const int n = grp == 0 ? 1 : 0;
            float*    x = xs + kTile * lastAt;
            float     vr[1] = {0.f}, vb[1] = {0.f};
            if(n && nLev > 1) take(RC, KC, lastAt);
            else if(n) {
                const float2 b = load2(lv[0].b, c.even);
                RC.rhs(c.red(b));
                KC.rhs(c.black(b));
            }
            first<1>(&RC, x + c.cr, vr, n);
            __syncthreads();
            for(int it = 0; it < coarsest; ++it) {
                if(it) {
                    half<1>(&RC, x + c.cr, c.offR, vr, vb, n);
                    __syncthreads();
                }
                half<1>(&KC, x + c.cb, -c.offR, vb, vr, n);
                __syncthreads();
            }
            for(int it = 0; it < coarsest; ++it) {
                if(it) {  // the black cells hold their solution already
                    half<1>(&KC, x + c.cb, -c.offR, vb, vr, n);
                    __syncthreads();
                }
                half<1>(&RC, x + c.cr, c.offR, vr, vb, n);
                __syncthreads();
            }
            if(n && nLev == 1) {
                store2(lv[0].x, c.even, c.cells(vr[0], vb[0]));
            }
        }
        for(int l = last - 1; l >= 1; --l) {
            const int S = (int)lv[l].nSlots;
            base -= S;
            if(last > 2 && l < last - 1) {  // the way down used the registers for a later level
                later(l, base);
                if(grp < S) {
                    const float2 b = load2(lv[l].b, grp * 512 + c.even);
                    R1[0].rhs(c.red(b));
                    K1[0].rhs(c.black(b));
                }
            }
            up<1>(R1, K1, c, xs + kTile * base, nb + base, S, grp);
        }
        if(nLev > 1) {
            up<2>(R0, K0, c, xs, nb, S0, grp);
#pragma unroll
            for(int q = 0; q < 2; ++q) {
                const int s = grp + 4 * q;
                if(s < S0) {
                    store2(lv[0].x, s * 512 + c.even, c.cells(xs[kTile * s + c.cr], xs[kTile * s + c.cb]));
                }
            }
        }
    }
};

}  // namespace bnn
