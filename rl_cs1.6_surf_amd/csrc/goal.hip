// goal.hip — the goal field: geodesic distance to a goal zone over the free
// voxels of an occupancy grid, and its trilinear sampler.
//
// Reference: python/surfgym/goalfield.py. build_goal_field (:159-298) seeds
// d = 0 on the free voxels of the inflated goal box, then relaxes
//   d[v] = min(d[v], d[v + o] + w_o)   for the 26 neighbour offsets o,
//   w_o = f32(cell * sqrt(|o|^2)), solid voxels pinned at +inf,
// in fp32 until nothing changes (:228-270), takes reach_max = the largest
// finite distance, replaces +inf by sentinel = reach_max + 2*cell, and stores
// round(d / (cell/8)) as uint16 (:272-297). GoalField.sample (:68-94)
// trilinearly interpolates the dequantised grid over its "honest" corners
// (value < reach_max + cell/2) only.
//
// Exactness. x -> fl(x + w) is monotone, so every relaxation order that runs
// until nothing changes ends at the same values: for each voxel, the least
// fp32 left-to-right sum of edge weights over the paths from a seed. The bake
// therefore relaxes in the order that suits the GPU instead of the
// reference's whole-grid Jacobi sweeps (one voxel of progress per sweep):
//
//   * 8x8x8 tiles, one wave per tile visit, are loaded with a one-voxel halo
//     into LDS and relaxed there until the tile is stable — a visit carries a
//     front across a tile;
//   * a tile writes back only the voxels it lowered, in place, and queues
//     the neighbour tiles whose halo holds one of them (a tile is stable
//     against its halo after a visit, so nothing else needs revisiting);
//   * sweeps consume one queue and fill the next, without the host; the
//     host reads the next queue's length every few sweeps and stops when it
//     is empty. Concurrent visits may read a halo value before or after a
//     neighbour lowers it: both are path sums, and any lowering after a read
//     queues the reader again, so an empty queue means every voxel is stable
//     against all 26 neighbours — the fixpoint.
//
// Work is proportional to the tiles the front crosses (times how often
// corrections re-cross them), not to grid size times path length.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/sdfr.h"

namespace {

thread_local char g_goal_err[256];

__attribute__((format(printf, 2, 3))) int32_t gfail(int32_t code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_goal_err, sizeof g_goal_err, fmt, ap);
    va_end(ap);
    return code;
}

constexpr int kT = 8;                    // tile edge (voxels)
constexpr int kTileVox = kT * kT * kT;
constexpr int kH = kT + 2;               // tile edge with halo
// LDS floats per column (8 and a gap) and per row of columns: 16-byte reads of
// 8 lanes along x fall 12 words apart, and 32 mod 64 from the next row's, so
// the 16 lanes of two rows read all 64 banks once.
constexpr int kCol = 12, kRow = 160;
constexpr int kTileLds = kH * kRow + 2 * kH * kH;
constexpr int kWaves = 4;                // tiles a block visits at once, one a wave
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxLocal = 96;            // local sweeps per visit; the tile is requeued if hit
constexpr int kSweepChunk = 32;          // sweeps launched between host checks
constexpr int64_t kPartMinTiles = 4096;  // grids of fewer tiles keep one queue (layout_of)
constexpr int kPartPitch = 32;           // words between the counts of 8 queues: a line each

// control words after the queues (uint32); the three counts are here while
// there is one queue, else in lines of their own (part_of)
enum { kCount0 = 0, kCount1 = 1, kCount2 = 2, kSeeds = 3, kReach = 4, kLastBusy = 5, kVisitsLo = 6,
       kVisitsHi = 7, kCtl = 8 };

struct GoalArgs {
    const uint8_t* occ;
    float* d;             // [tiles][y][x][z], kTileVox a tile; +inf past the grid's edge
    uint64_t* open;       // [tiles][kT]: plane z's free voxels inside the grid, bit 8 * y + x
    uint32_t* mark;       // [tiles] last sweep the tile was queued for
    uint32_t* queues;     // [2][parts][part_cap], sweep k reads [k & 1]
    uint32_t* counts;     // [3][parts], part_pitch words apart: sweep k's is [k % 3]
    int parts;            // queues a sweep's tiles are split into: 8, one per XCD, or 1
    uint32_t part_cap, part_pitch;
    uint32_t* ctl;        // [kCtl]
    int nx, ny, nz;
    int tx, ty, tz;       // tiles per axis
    uint32_t tiles;
    float w1, w2, w3;     // edge weights for |o|^2 = 1, 2, 3
};

// Which of 8 queues a tile goes to. A tile's halo lies in its neighbours'
// lines, so near tiles are kept in one queue, whose sweep blocks run on one
// XCD (block b on XCD b % 8) and share its L2:
// blocks of 4 x 2 x 2 tiles, dealt out in order over rows made odd in length,
// so that neighbours along every axis go to different queues.
__device__ __forceinline__ uint32_t part_of(const GoalArgs& a, int tx, int ty, int tz) {
    if (a.parts == 1) return 0u;
    const uint32_t sx = (uint32_t)((a.tx + 3) >> 2) | 1u, sy = (uint32_t)((a.ty + 1) >> 1);
    return (((uint32_t)(tz >> 1) * sy + (uint32_t)(ty >> 1)) * sx + (uint32_t)(tx >> 2)) & 7u;
}

__device__ __forceinline__ uint32_t* count_of(const GoalArgs& a, uint32_t k, uint32_t part) {
    return a.counts + ((k % 3u) * (uint32_t)a.parts + part) * a.part_pitch;
}

__device__ __forceinline__ uint32_t* queue_of(const GoalArgs& a, uint32_t k, uint32_t part) {
    return a.queues + ((size_t)(k & 1u) * a.parts + part) * a.part_cap;
}

// Block b runs on XCD b % 8. Kernels that walk the whole grid give each XCD a
// contiguous eighth of their n items, as a line of the grid's rows holds several
// tiles' voxels and is best read and written through one L2 (268 M voxels:
// goal_init 480 -> 360 to 397 us, goal_quantise 650 -> 561). The launch is a
// multiple of 8 blocks.
__device__ __forceinline__ uint32_t xcd_share(uint32_t n) { return (n + 7) / 8; }

// d = +inf everywhere, 0 on the free voxels of the seed box; the tiles that
// hold a seed or touch one through their halo form the first queue. Tiles
// without a free voxel are marked as if queued for good: no visit could lower
// anything there. A wave a tile. A lane reads one of the tile's 64 rows, eight
// bytes at once, whose free voxels are a byte of the tile's masks as they lie;
// its column's seeds it takes from the rows' lanes, in the seed box's tiles
// only. What bounds it is the bytes: 268 M voxels QQINIT us (700 with a byte a
// lane and column, 370 a voxel a thread).
__global__ __launch_bounds__(256) void goal_init(GoalArgs a, int lx, int ly, int lz, int hx, int hy,
                                                 int hz, int tlx, int tly, int tlz, int thx, int thy,
                                                 int thz) {
    const int lane = threadIdx.x & 63;
    uint32_t seeds = 0;
    const uint32_t share = xcd_share((a.tiles + 3) / 4);
    for (uint32_t i = blockIdx.x >> 3; i < share; i += gridDim.x >> 3) {
        const uint32_t t = ((blockIdx.x & 7u) * share + i) * 4 + (threadIdx.x >> 6);
        if (t >= a.tiles) break;
        const int tx = (int)(t % (uint32_t)a.tx);
        const uint32_t r = t / (uint32_t)a.tx;
        const int ty = (int)(r % (uint32_t)a.ty), tz = (int)(r / (uint32_t)a.ty);
        const int x0 = tx * kT, y0 = ty * kT, z0 = tz * kT;
        uint64_t solid = ~0ull;   // bytes of row (z0 + lane / 8, y0 + lane % 8)
        const int ry = y0 + (lane & 7), rz = z0 + (lane >> 3);
        if (ry < a.ny && rz < a.nz) {
            const uint8_t* o = a.occ + ((int64_t)rz * a.ny + ry) * a.nx + x0;
            if (x0 + kT <= a.nx) {
                __builtin_memcpy(&solid, o, 8);   // (at any alignment)
            } else {
                for (int b = 0; b < a.nx - x0; ++b)
                    if (o[b] == 0) solid &= ~(0xffull << (8 * b));
            }
        }
        // bit i: byte i is zero (the top bit of every non-zero byte, gathered)
        const uint64_t low = 0x7f7f7f7f7f7f7f7full;
        const uint64_t some = (((solid & low) + low) | solid) & ~low;
        const uint32_t free = (uint32_t)((((some >> 7) * 0x0102040810204080ull) >> 56) ^ 0xffull);
        ((uint8_t*)(a.open + (int64_t)t * kT))[lane] = (uint8_t)free;
        const bool any = __any(free != 0u);
        const bool in = tx >= tlx && tx <= thx && ty >= tly && ty <= thy && tz >= tlz && tz <= thz;
        float v[kT];
#pragma unroll
        for (int z = 0; z < kT; ++z) v[z] = INFINITY;
        if (in) {   // uniform
            const int x = x0 + (lane & 7), y = y0 + (lane >> 3);
            const bool box = x >= lx && x <= hx && y >= ly && y <= hy;
#pragma unroll
            for (int z = 0; z < kT; ++z) {
                const uint32_t row = __shfl(free, z * kT + (lane >> 3));
                const bool seed = box && z0 + z >= lz && z0 + z <= hz && ((row >> (lane & 7)) & 1u) != 0u;
                if (seed) v[z] = 0.0f;
                seeds += seed;
            }
        }
        float4* col = (float4*)(a.d + (int64_t)t * kTileVox + lane * kT);
        col[0] = make_float4(v[0], v[1], v[2], v[3]);
        col[1] = make_float4(v[4], v[5], v[6], v[7]);
        if (lane == 0) {
            a.mark[t] = !any ? ~0u : in ? 1u : 0u;
            if (in && any) {
                const uint32_t part = part_of(a, tx, ty, tz);
                queue_of(a, 1u, part)[atomicAdd(count_of(a, 1u, part), 1u)] = t;
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) seeds += __shfl_down(seeds, off);
    if (lane == 0 && seeds) atomicAdd(&a.ctl[kSeeds], seeds);
}

// The smaller of two distances: of non-negative floats (+inf among them) as
// their bit patterns order, which spares the compiler the quieting of NaNs.
__device__ __forceinline__ float least(float a, float b) {
    return __uint_as_float(min(__float_as_uint(a), __float_as_uint(b)));
}

// Lane masks of a tile's columns (lane = 8 * y + x): those on its low / any /
// high side along x and along y.
__device__ __forceinline__ uint64_t side_x(int d) {
    return d < 0 ? 0x0101010101010101ull : d > 0 ? 0x8080808080808080ull : ~0ull;
}
__device__ __forceinline__ uint64_t side_y(int d) {
    return d < 0 ? 0xffull : d > 0 ? 0xffull << 56 : ~0ull;
}

// Orders a wave's LDS writes before its later reads (one wave owns the tile,
// and its LDS operations execute in order).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sweep k: visit every tile queued for it, queue tiles for sweep k + 1, clear
// the counts of sweep k + 2 (those of sweep k - 1).
//
// One wave visits one tile, a lane per (x, y) column with its 8 voxels in
// registers. The 10 x 10 columns with the halo lie in LDS, z fastest, so a
// relaxation reads each of a column's 8 neighbour columns with two 16-byte
// loads. x -> fl(x + w) is monotone, so fl(min(a, b) + w) = min(fl(a + w),
// fl(b + w)): the four face columns and the four edge columns are reduced
// before their weights are added (2 wide LDS reads and ~17 vector
// instructions a voxel instead of 26 and 52). Up and down its own column a
// lane relaxes in order, so a value crosses the tile along z in one pass.
//
// The distances lie tile by tile, each column's 8 voxels together, so a lane
// takes a column in two 16-byte loads (8 loads a visit with the halo, ~100
// lines; rows of the grid took 28 loads and 240 lines), and the free voxels
// are lane masks in scalar registers.
//
// What bounds it: the time of the slowest visits. In a bake of a closed scene of
// 256x256x128 voxels (50 sweeps, up to 23 us each) no unit is near its limit in
// any sweep: vector issue is busy 28% of the cycles at most and LDS 14% (a sixth
// of it conflicts). In the ~20 long sweeps (up to 5000 visits, one a wave) a wave
// spends 42% of its time waiting for memory and LDS and 31% for its turn at the
// SIMD, over the ~10 relaxations of a visit; in the ~30 short ones it is the
// chain of round trips to memory of one visit (queue, tile, mark, slot: ~6 us).
// 29 us a sweep with a block of 512 threads and 26 LDS reads a voxel, 18 with a
// wave a tile, 16 with the columns loaded straight to their lanes; a whole bake
// of that scene 1086 us with a queue per XCD, 887 with the distances by tile, 840
// to 917 by run with the halo's loads under a branch and the pass down z as
// selects. Also measured: flags per tile instead of queues (no claims, but a
// static deal of tiles to waves: 28 us a sweep), reading a mark before its atomic
// (+2 us), no order along z (+2 us), queueing only tiles whose halo copy would
// fall (20% fewer visits, each 3 us longer).
__global__ __launch_bounds__(kThreads) void goal_sweep(GoalArgs a, const uint64_t* __restrict__ open_planes,
                                                       uint32_t k) {
    __shared__ __align__(16) float s_all[kWaves][kTileLds];
    const uint32_t part = blockIdx.x % (uint32_t)a.parts, block = blockIdx.x / (uint32_t)a.parts;
    const uint32_t blocks = gridDim.x / (uint32_t)a.parts;   // of this queue
    const uint32_t* qi = queue_of(a, k, part);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // consecutive tiles go to different blocks: a short queue spreads over the
    // GPU. The first entry is read with the length, not after it (an entry
    // past the queue's end is not used).
    uint32_t e = (uint32_t)wave * blocks + block;
    uint32_t tile_v = e < a.part_cap ? qi[e] : 0u;
    const uint32_t n = *count_of(a, k, part);
    if (block == 0 && threadIdx.x == 0) {
        *count_of(a, k + 2u, part) = 0u;
        if (n) {
            a.ctl[kLastBusy] = k;
            atomicAdd((unsigned long long*)&a.ctl[kVisitsLo], (unsigned long long)n);
        }
    }
    const int lx = lane & 7, ly = lane >> 3;
    float* s = s_all[wave];
    float* zlo = s + kH * kRow;         // the halo planes below and above
    float* zhi = zlo + kH * kH;
    const int c = (ly + 1) * kH + (lx + 1);
    float* own = s + (ly + 1) * kRow + (lx + 1) * kCol;
    const float w1 = a.w1, w2 = a.w2, w3 = a.w3;
    // lanes 0..35 also load a halo column each: the sides x = -1, x = 8,
    // y = -1, y = 8 (8 lanes each), then the corners
    const int side = lane >> 3, at = (lane & 7) + 1;
    const int rx = side == 0 ? 0 : side == 1 ? kH - 1 : side > 3 ? (lane & 1) * (kH - 1) : at;
    const int ry = side == 2 ? 0 : side == 3 ? kH - 1 : side > 3 ? ((lane >> 1) & 1) * (kH - 1) : at;
    float* ring = s + ry * kRow + rx * kCol;
    // ... from the tile its column lies in
    const int rtx = rx == 0 ? -1 : rx == kH - 1 ? 1 : 0, rty = ry == 0 ? -1 : ry == kH - 1 ? 1 : 0;
    const int rcol = ((ry - 1) & 7) * kT + ((rx - 1) & 7);
    const int64_t layer = (int64_t)a.tx * a.ty * kTileVox;   // distances to the tile above
    const int64_t roff = ((int64_t)rty * a.tx + rtx) * kTileVox + rcol * kT;
    for (; e < n; e += blocks * kWaves, tile_v = e < n ? qi[e] : 0u) {
        const uint32_t tile = __builtin_amdgcn_readfirstlane(tile_v);
        const int tx = (int)(tile % (uint32_t)a.tx);
        const uint32_t r = tile / (uint32_t)a.tx;
        const int ty = (int)(r % (uint32_t)a.ty), tz = (int)(r / (uint32_t)a.ty);
        const bool on_ring = lane < 36 && tx + rtx >= 0 && tx + rtx < a.tx && ty + rty >= 0 && ty + rty < a.ty;
        // the lane's own column and its halo column, both with the voxels
        // below and above; outside the grid nothing lowers a neighbour
        float* home = a.d + (int64_t)tile * kTileVox + lane * kT;
        const float* rim = a.d + (int64_t)tile * kTileVox + roff;
        const float4 c0 = ((const float4*)home)[0], c1 = ((const float4*)home)[1];
        // (under a branch: as a choice of values the compiler chooses between
        // addresses, one on the stack, and loads through the flat path)
        float4 r0 = make_float4(INFINITY, INFINITY, INFINITY, INFINITY), r1 = r0;
        if (on_ring) {
            r0 = ((const float4*)rim)[0];
            r1 = ((const float4*)rim)[1];
        }
        float cb = INFINITY, ca = INFINITY, rb = INFINITY, ra = INFINITY;
        if (tz > 0) {   // uniform
            cb = home[kT - 1 - layer];
            if (on_ring) rb = rim[kT - 1 - layer];
        }
        if (tz + 1 < a.tz) {
            ca = home[layer];
            if (on_ring) ra = rim[layer];
        }
        const float cv[kT] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        uint64_t open[kT];
#pragma unroll
        for (int z = 0; z < kT; ++z) open[z] = open_planes[(int64_t)tile * kT + z];
        float start[kT], cur[kT];
#pragma unroll
        for (int z = 0; z < kT; ++z) start[z] = cur[z] = cv[z];
        *(float4*)own = c0;
        *(float4*)(own + 4) = c1;
        zlo[c] = cb;
        zhi[c] = ca;
        if (lane < 36) {
            *(float4*)ring = r0;
            *(float4*)(ring + 4) = r1;
            zlo[ry * kH + rx] = rb;
            zhi[ry * kH + rx] = ra;
        }
        wave_sync();
        // what the planes below and above give the first and last voxel
        // (the halo does not change during a visit)
        auto beside = [&](const float* p) {
            const float f = least(least(p[c - 1], p[c + 1]), least(p[c - kH], p[c + kH]));
            const float g = least(least(p[c - kH - 1], p[c - kH + 1]), least(p[c + kH - 1], p[c + kH + 1]));
            return least(least(f + w2, g + w3), p[c] + w1);
        };
        const float below = beside(zlo), above = beside(zhi);
        // a pass in which no voxel lowered saw a constant tile: it is stable
        bool moving = true;
        for (int it = 0; moving && it < kMaxLocal; ++it) {
            float f[kT], g[kT];
            auto column = [&](int o, float* m, bool first) {
                const float4 lo = *(const float4*)(own + o), hi = *(const float4*)(own + o + 4);
                const float q[kT] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                for (int z = 0; z < kT; ++z) m[z] = first ? q[z] : least(m[z], q[z]);
            };
            column(-kCol, f, true);
            column(kCol, f, false);
            column(-kRow, f, false);
            column(kRow, f, false);
            column(-kRow - kCol, g, true);
            column(-kRow + kCol, g, false);
            column(kRow - kCol, g, false);
            column(kRow + kCol, g, false);
            // by the voxels above and below: Q the neighbour columns' share,
            // and the column's own
            float q[kT], m[kT];
#pragma unroll
            for (int z = 0; z < kT; ++z) q[z] = least(least(f[z] + w2, g[z] + w3), cur[z] + w1);
#pragma unroll
            for (int z = 0; z < kT; ++z) {
                m[z] = least(least(cur[z], least(f[z] + w1, g[z] + w2)),
                             least(z ? q[z - 1] : below, z < kT - 1 ? q[z + 1] : above));
                if (z) m[z] = least(m[z], m[z - 1] + w1);
                m[z] = __builtin_amdgcn_inverse_ballot_w64(open[z]) ? m[z] : INFINITY;
            }
#pragma unroll
            for (int z = kT - 2; z >= 0; --z) {
                const float down = least(m[z], m[z + 1] + w1);
                m[z] = __builtin_amdgcn_inverse_ballot_w64(open[z]) ? down : INFINITY;
            }
            bool lowered = false;
#pragma unroll
            for (int z = 0; z < kT; ++z) {
                lowered |= m[z] < cur[z];
                cur[z] = m[z];
            }
            moving = __any(lowered);
            if (lowered) {
                *(float4*)own = make_float4(cur[0], cur[1], cur[2], cur[3]);
                *(float4*)(own + 4) = make_float4(cur[4], cur[5], cur[6], cur[7]);
            }
            wave_sync();
        }
        bool any = false;
#pragma unroll
        for (int z = 0; z < kT; ++z) any |= cur[z] < start[z];
        if (any) {   // no other wave writes this tile in this sweep
            ((float4*)home)[0] = make_float4(cur[0], cur[1], cur[2], cur[3]);
            ((float4*)home)[1] = make_float4(cur[4], cur[5], cur[6], cur[7]);
        }
        // neighbour tiles whose halo holds a lowered voxel; lane t < 27 looks
        // after direction t
        const uint64_t b0 = __ballot(any), bl = __ballot(cur[0] < start[0]), bh = __ballot(cur[kT - 1] < start[kT - 1]);
        const int dz = lane / 9 - 1, dy = (lane / 3) % 3 - 1, dx = lane % 3 - 1;
        bool push = ((dz < 0 ? bl : dz > 0 ? bh : b0) & side_x(dx) & side_y(dy)) != 0;
        if (lane == 13) push = moving;   // the local cap was hit: visit this one again
        if (lane < 27 && push) {
            const int ux = tx + dx, uy = ty + dy, uz = tz + dz;
            if (ux >= 0 && uy >= 0 && uz >= 0 && ux < a.tx && uy < a.ty && uz < a.tz) {
                const uint32_t u = ((uint32_t)uz * (uint32_t)a.ty + (uint32_t)uy) * (uint32_t)a.tx + (uint32_t)ux;
                if (atomicMax(&a.mark[u], k + 1u) <= k) {
                    const uint32_t to = part_of(a, ux, uy, uz);
                    queue_of(a, k + 1u, to)[atomicAdd(count_of(a, k + 1u, to), 1u)] = u;
                }
            }
        }
    }
}

// reach_max: the largest finite distance (non-negative floats order as their
// bit patterns). Four distances per load over whole tiles (+inf past the
// grid's edge); one atomic per block (atomics from every wave to the one word
// serialise).
constexpr int kReachBlocks = 512;
__global__ __launch_bounds__(256) void goal_reach_max(GoalArgs a) {
    __shared__ uint32_t s_m[4];
    uint32_t m = 0;
    const int64_t n4 = (int64_t)a.tiles * (kTileVox / 4);
    const float4* d4 = reinterpret_cast<const float4*>(a.d);
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += step) {
        const float4 v = d4[i];
        if (v.x != INFINITY) m = max(m, __float_as_uint(v.x));
        if (v.y != INFINITY) m = max(m, __float_as_uint(v.y));
        if (v.z != INFINITY) m = max(m, __float_as_uint(v.z));
        if (v.w != INFINITY) m = max(m, __float_as_uint(v.w));
    }
    for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_down(m, off));
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(s_m[0], s_m[1]), max(s_m[2], s_m[3]));
        if (m) atomicMax(a.ctl + kReach, m);
    }
}

// +inf -> sentinel, then round(d / quant) clamped to [0, 65535]. The
// reference divides a CUDA tensor by a Python scalar, which torch evaluates as
// d * (1/quant) with the reciprocal rounded to fp32 (identical to d / quant
// for the power-of-two cells the reference picks), and rounds half to even.
// The sentinel is the host's reach_max + 2*cell, from the largest distance
// goal_reach_max left; a field beyond the uint16 range writes nothing. A block
// turns four tiles along x into rows of 32 voxels through LDS (rows 36 words
// apart: the 64 columns of a wave then fall on 64 banks), so that both
// outputs are written in whole lines, four voxels a thread (`wide`: rows and
// outputs are aligned for it) or one beside the next (801x803x203 voxels 256 us;
// 272 a voxel a thread from rows of the grid). 268 M voxels 561 to 580 us by run.
__global__ __launch_bounds__(256) void goal_quantise(GoalArgs a, double cell, float inv_quant, float quant,
                                                     uint16_t* q_out, float* g_out, int wide) {
    constexpr int kSpan = 4 * kT, kPitch = kSpan + 4;
    __shared__ __align__(16) float s[kT * kT * kPitch];
    const double sentinel_d = (double)__uint_as_float(a.ctl[kReach]) + 2.0 * cell;
    if (sentinel_d / (cell / 8.0) > 65535.0) return;
    const float sentinel = (float)sentinel_d;
    auto code = [&](float v) {
        if (v == INFINITY) v = sentinel;
        return (uint16_t)fminf(fmaxf(rintf(v * inv_quant), 0.0f), 65535.0f);
    };
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t spans = (uint32_t)(a.tx + 3) / 4u, groups = spans * (uint32_t)a.ty * (uint32_t)a.tz;
    const uint32_t share = xcd_share(groups);
    for (uint32_t i = blockIdx.x >> 3; i < share; i += gridDim.x >> 3) {
        const uint32_t gr = (blockIdx.x & 7u) * share + i;
        if (gr >= groups) break;   // (uniform)
        const uint32_t row = gr / spans;   // of tiles: tz * ty_count + ty
        const int tx0 = (int)(gr - row * spans) * 4;
        const int ty = (int)(row % (uint32_t)a.ty), tz = (int)(row / (uint32_t)a.ty);
        if (tx0 + wave < a.tx) {
            const float4* col = (const float4*)(a.d + ((int64_t)row * a.tx + tx0 + wave) * kTileVox + lane * kT);
            const float4 lo = col[0], hi = col[1];
            const float v[kT] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int z = 0; z < kT; ++z) s[(z * kT + (lane >> 3)) * kPitch + wave * kT + (lane & 7)] = v[z];
        }
        __syncthreads();
        // line l of the LDS is the row (tz * 8 + l / 8, ty * 8 + l % 8)
        auto place = [&](int line, int c) -> int64_t {   // of its voxel c; -1 outside the grid
            const int x = tx0 * kT + c, y = ty * kT + (line & 7), z = tz * kT + (line >> 3);
            return x < a.nx && y < a.ny && z < a.nz ? ((int64_t)z * a.ny + y) * a.nx + x : -1;
        };
        if (wide) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int line = j * 32 + (int)(threadIdx.x >> 3), c = (int)(threadIdx.x & 7) * 4;
                const int64_t at = place(line, c);
                if (at < 0) continue;
                const float4 f = *(const float4*)(s + line * kPitch + c);
                const ushort4 u = make_ushort4(code(f.x), code(f.y), code(f.z), code(f.w));
                if (q_out) *(ushort4*)(q_out + at) = u;
                if (g_out)
                    *(float4*)(g_out + at) =
                        make_float4((float)u.x * quant, (float)u.y * quant, (float)u.z * quant, (float)u.w * quant);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int line = j * 8 + (int)(threadIdx.x >> 5), c = (int)(threadIdx.x & 31);
                const int64_t at = place(line, c);
                if (at < 0) continue;
                const uint16_t u = code(s[line * kPitch + c]);
                if (q_out) q_out[at] = u;
                if (g_out) g_out[at] = (float)u * quant;
            }
        }
        __syncthreads();
    }
}

// GoalField.sample (goalfield.py:68-94): trilinear over the honest corners.
struct FieldArgs {
    const void* grid;
    float quant;
    int nx, ny, nz;
    double mnx, mny, mnz, cell;
    float valid_max, sentinel;
};

template <int GRID>
__device__ __forceinline__ float field_at(const FieldArgs& a, double px, double py, double pz) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const double gx = (px - a.mnx) / a.cell - 0.5;
    const double gy = (py - a.mny) / a.cell - 0.5;
    const double gz = (pz - a.mnz) / a.cell - 0.5;
    const double fx0 = floor(gx), fy0 = floor(gy), fz0 = floor(gz);
    const float fx = (float)(gx - fx0), fy = (float)(gy - fy0), fz = (float)(gz - fz0);
    // corner indices clamped in double: a far-off position cannot overflow
    const double cx[2] = {fmin(fmax(fx0, 0.0), nx - 1.0), fmin(fmax(fx0 + 1.0, 0.0), nx - 1.0)};
    const double cy[2] = {fmin(fmax(fy0, 0.0), ny - 1.0), fmin(fmax(fy0 + 1.0, 0.0), ny - 1.0)};
    const double cz[2] = {fmin(fmax(fz0, 0.0), nz - 1.0), fmin(fmax(fz0 + 1.0, 0.0), nz - 1.0)};
    float num = 0.0f, den = 0.0f;
#pragma unroll
    for (int dz = 0; dz < 2; ++dz)
#pragma unroll
        for (int dy = 0; dy < 2; ++dy)
#pragma unroll
            for (int dx = 0; dx < 2; ++dx) {
                const int64_t k = ((int64_t)cz[dz] * ny + (int64_t)cy[dy]) * nx + (int64_t)cx[dx];
                const float v = GRID == SDFR_F32 ? ((const float*)a.grid)[k]
                                                 : (float)((const uint16_t*)a.grid)[k] * a.quant;
                const float wx = dx ? fx : 1.0f - fx;
                const float wy = dy ? fy : 1.0f - fy;
                const float wz = dz ? fz : 1.0f - fz;
                const float w = ((wx * wy) * wz) * (v < a.valid_max ? 1.0f : 0.0f);
                num = num + w * v;
                den = den + w;
            }
    return den > 1e-6f ? num / fmaxf(den, 1e-6f) : a.sentinel;
}

template <int POS>
__device__ __forceinline__ double pos_at(const void* pos, int64_t i) {
    return POS == SDFR_F64 ? ((const double*)pos)[i] : (double)((const float*)pos)[i];
}

template <int GRID, int POS>
__global__ __launch_bounds__(256) void goal_sample(FieldArgs a, const void* __restrict__ pos, int64_t pos_stride,
                                                   int64_t n, float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t o = i * pos_stride;
    out[i] = field_at<GRID>(a, pos_at<POS>(pos, o), pos_at<POS>(pos, o + 1), pos_at<POS>(pos, o + 2));
}

// GoalField.descent_yaw (goalfield.py:101-107): the yaw of the steepest
// horizontal descent from samples one cell off along +x, -x, +y and -y. What
// bounds it at a reservoir's ~1500 positions is launches and round trips to
// memory, so one launch does what took fifteen (positions to float64, four
// offset copies, samples, differences, atan2, degrees, remainder): four lanes
// a position, one sample each, handed over by shuffles, so a position's 32
// gathers are in flight together. 1500 host positions: 108 us a call before,
// 42 now, most of it the copies there and back.
template <int GRID, int POS>
__global__ __launch_bounds__(256) void goal_yaw(FieldArgs a, const void* __restrict__ pos, int64_t pos_stride,
                                                int64_t n, float* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, i = t >> 2;
    const int dir = (int)(t & 3);
    // lanes past the end sample the last position: the shuffles want every lane
    const int64_t o = (i < n ? i : n - 1) * pos_stride;
    const double h = dir & 1 ? -a.cell : a.cell;
    const double px = pos_at<POS>(pos, o) + (dir < 2 ? h : 0.0);
    const double py = pos_at<POS>(pos, o + 1) + (dir < 2 ? 0.0 : h);
    const float s = field_at<GRID>(a, px, py, pos_at<POS>(pos, o + 2));
    const float diff = s - __shfl_down(s, 1);   // lane 0 of 4: along x, lane 2: along y
    const float dx = diff, dy = __shfl_down(diff, 2);
    if (dir != 0 || i >= n) return;
    float yaw = fmodf(atan2f(-dy, -dx) * 57.29577951308232f, 360.0f);   // degrees, Python's remainder
    if (yaw < 0.0f) yaw += 360.0f;
    out[i] = yaw;
}

constexpr int64_t kCountWords = 3 * 8 * kPartPitch;   // of eight queues

struct Layout {
    int64_t d_off, open_off, mark_off, q_off, ctl_off, total;
    int64_t part_cap;   // tiles a queue holds
    int parts;
    uint32_t tiles;
};

Layout layout_of(int nx, int ny, int nz) {
    Layout l;
    const int64_t tiles = (int64_t)((nx + kT - 1) / kT) * ((ny + kT - 1) / kT) * ((nz + kT - 1) / kT);
    l.tiles = (uint32_t)tiles;
    // eight queues where there are tiles enough to keep them even, each with
    // room for an eighth of the blocks that part_of deals out, whole or not. A
    // single queue's count is one address that every visit's pushes wait for:
    // 12 ns a visit, 3 with eight queues (4096x4096x1 voxels, a quarter solid:
    // 162 ms a bake with one queue, 35 with eight).
    const int64_t tx = (nx + kT - 1) / kT, ty = (ny + kT - 1) / kT, tz = (nz + kT - 1) / kT;
    l.parts = tiles >= kPartMinTiles ? 8 : 1;
    l.part_cap = l.parts == 8 ? ((((tx + 3) / 4) | 1) * ((ty + 1) / 2) * ((tz + 1) / 2) + 7) / 8 * 16 : tiles;
    l.d_off = 0;
    l.open_off = l.d_off + tiles * kTileVox * 4;
    l.mark_off = l.open_off + tiles * kT * 8;
    l.q_off = l.mark_off + tiles * 4;
    // two sweeps' queues, then (eight queues) their counts right before the
    // control words
    l.ctl_off = l.q_off + (2 * l.parts * l.part_cap + (l.parts == 8 ? kCountWords : 0)) * 4;
    l.ctl_off = (l.ctl_off + 63) & ~(int64_t)63;
    l.total = l.ctl_off + kCtl * 4;
    return l;
}

}  // namespace

extern "C" {

SDFR_API const char* sdfr_goal_last_error(void) { return g_goal_err; }

SDFR_API int64_t sdfr_goal_workspace_bytes(int32_t nx, int32_t ny, int32_t nz) {
    if (nx <= 0 || ny <= 0 || nz <= 0) return -2;
    return layout_of(nx, ny, nz).total;
}

SDFR_API int32_t sdfr_goal_bake(const uint8_t* occ, int32_t nx, int32_t ny, int32_t nz, float cell,
                                const int32_t* seed_lo, const int32_t* seed_hi, int32_t max_sweeps,
                                uint16_t* grid_q, float* grid, SdfrGoalInfo* info, void* workspace,
                                int64_t workspace_size, void* stream) {
    g_goal_err[0] = '\0';
    if (!occ || !seed_lo || !seed_hi || !workspace || !info || (!grid_q && !grid))
        return gfail(-1, "sdfr_goal_bake: null pointer argument");
    if (nx <= 0 || ny <= 0 || nz <= 0)
        return gfail(-2, "sdfr_goal_bake: grid dims must be positive (got %d x %d x %d)", nx, ny, nz);
    if (!(cell > 0.0f) || !isfinite(cell)) return gfail(-2, "sdfr_goal_bake: cell must be positive");
    if (max_sweeps <= 0) return gfail(-2, "sdfr_goal_bake: max_sweeps must be positive");
    const int64_t tiles64 = (int64_t)((nx + kT - 1) / kT) * ((ny + kT - 1) / kT) * ((nz + kT - 1) / kT);
    if (tiles64 > 0x3fffffffLL) return gfail(-2, "sdfr_goal_bake: grid too large");
    const Layout L = layout_of(nx, ny, nz);
    if (workspace_size < L.total)
        return gfail(-2, "sdfr_goal_bake: workspace of %lld bytes needed (got %lld)",
                     (long long)L.total, (long long)workspace_size);
    if (((uintptr_t)workspace & 63u) != 0)
        return gfail(-2, "sdfr_goal_bake: workspace must be 64-byte aligned");
    // the seed box, clipped to the grid (goalfield.py:228-240)
    const int dims[3] = {nx, ny, nz};
    int lo[3], hi[3], tlo[3], thi[3];
    for (int j = 0; j < 3; ++j) {
        lo[j] = seed_lo[j] < 0 ? 0 : seed_lo[j];
        hi[j] = seed_hi[j] > dims[j] - 1 ? dims[j] - 1 : seed_hi[j];
        if (hi[j] < lo[j])
            return gfail(-5, "sdfr_goal_bake: goal zone contains no free voxel (empty seed box)");
        const int ntj = (dims[j] + kT - 1) / kT;
        tlo[j] = lo[j] == 0 ? 0 : (lo[j] - 1) / kT;
        thi[j] = (hi[j] + 1) / kT > ntj - 1 ? ntj - 1 : (hi[j] + 1) / kT;
    }
    hipStream_t st = (hipStream_t)stream;
    uint8_t* ws = (uint8_t*)workspace;
    GoalArgs g;
    g.occ = occ;
    g.d = (float*)(ws + L.d_off);
    g.open = (uint64_t*)(ws + L.open_off);
    g.mark = (uint32_t*)(ws + L.mark_off);
    g.queues = (uint32_t*)(ws + L.q_off);
    g.ctl = (uint32_t*)(ws + L.ctl_off);
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    g.tx = (nx + kT - 1) / kT;
    g.ty = (ny + kT - 1) / kT;
    g.tz = (nz + kT - 1) / kT;
    g.tiles = L.tiles;
    // cell * sqrt(|o|^2) in float64 (Python floats), added to an fp32 tensor
    // as an fp32 scalar
    g.w1 = (float)((double)cell * sqrt(1.0));
    g.w2 = (float)((double)cell * sqrt(2.0));
    g.w3 = (float)((double)cell * sqrt(3.0));
    g.parts = L.parts;
    g.part_cap = (uint32_t)L.part_cap;
    g.part_pitch = g.parts == 8 ? kPartPitch : 1;
    g.counts = g.parts == 8 ? g.ctl - kCountWords : g.ctl + kCount0;
    const int64_t shared = (g.parts == 8 ? kCountWords : 0) + kCtl;   // words the host reads
    uint32_t host[kCountWords + kCtl];
    uint32_t* const host_ctl = host + (shared - kCtl);
    uint32_t* const host_counts = g.parts == 8 ? host : host_ctl + kCount0;
    memset(host, 0, sizeof host);
    uint32_t* const dev_words = g.ctl - (shared - kCtl);
    hipError_t e = hipMemcpyAsync(dev_words, host, shared * 4, hipMemcpyHostToDevice, st);
    if (e != hipSuccess) return gfail(-4, "sdfr_goal_bake: %s", hipGetErrorString(e));
    const uint32_t quads = (L.tiles + 3) / 4;   // four tiles a block
    const int init_blocks = (int)(quads > 8192 ? 8192 : (quads + 7) / 8 * 8);
    goal_init<<<init_blocks, 256, 0, st>>>(g, lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], tlo[0], tlo[1],
                                           tlo[2], thi[0], thi[1], thi[2]);
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cus = 256;
    const int sweep_blocks = cus * 5 / 8 * 8 > 0 ? cus * 5 / 8 * 8 : 8;   // 5 a CU fit its registers; a multiple of the queues
    uint32_t k = 1;
    bool done = false;
    while (!done && (int64_t)k <= max_sweeps) {
        for (int j = 0; j < kSweepChunk && (int64_t)k <= max_sweeps; ++j, ++k)
            goal_sweep<<<sweep_blocks, kThreads, 0, st>>>(g, g.open, k);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(host, dev_words, shared * 4, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return gfail(-4, "sdfr_goal_bake: %s", hipGetErrorString(e));
        if (host_ctl[kSeeds] == 0)
            return gfail(-5, "sdfr_goal_bake: goal zone contains no free voxel");
        done = true;   // k is the next sweep: are its queues empty?
        for (int p = 0; p < g.parts; ++p)
            if (host_counts[((k % 3u) * g.parts + p) * g.part_pitch]) done = false;
    }
    if (!done) return gfail(-7, "sdfr_goal_bake: not converged after %d sweeps", max_sweeps);
    goal_reach_max<<<kReachBlocks, 256, 0, st>>>(g);
    const double quant = (double)cell / 8.0;
    const float quant_f = (float)quant;
    const float inv_quant = 1.0f / quant_f;
    const int wide = nx % 4 == 0 && ((uintptr_t)grid_q & 7u) == 0 && ((uintptr_t)grid & 15u) == 0;
    const int64_t groups = (int64_t)((g.tx + 3) / 4) * g.ty * g.tz;
    const int quantise_blocks = (int)(groups > 65536 ? 65536 : (groups + 7) / 8 * 8);
    goal_quantise<<<quantise_blocks, 256, 0, st>>>(g, (double)cell, inv_quant, quant_f, grid_q, grid, wide);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(host_ctl, g.ctl, kCtl * 4, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return gfail(-4, "sdfr_goal_bake: %s", hipGetErrorString(e));
    float reach_max;
    memcpy(&reach_max, &host_ctl[kReach], 4);
    // Python floats: sentinel = reach_max + 2*cell, quant = cell/8; stored fp32
    const double sentinel = (double)reach_max + 2.0 * (double)cell;
    info->reach_max = reach_max;
    info->sentinel = (float)sentinel;
    info->quant = quant_f;
    info->sweeps = (int32_t)host_ctl[kLastBusy];
    info->n_seed = (int64_t)host_ctl[kSeeds];
    info->tile_visits = (int64_t)host_ctl[kVisitsLo] | ((int64_t)host_ctl[kVisitsHi] << 32);
    if (sentinel / quant > 65535.0)
        return gfail(-6, "sdfr_goal_bake: sentinel %.0fu exceeds the uint16 range at quant %gu",
                     sentinel, quant);
    return 0;
}

// The checks that goal_sample and goal_yaw share; fills `a`.
static int32_t field_args(const char* fn, FieldArgs* a, const void* grid, int32_t grid_dtype, float quant, int32_t nx,
                          int32_t ny, int32_t nz, const double* mins, double cell, double reach_max, const void* pos,
                          int32_t pos_dtype, int64_t pos_stride, int64_t n, const float* out, int per_block) {
    g_goal_err[0] = '\0';
    if (!grid || !mins || !out || (!pos && n > 0)) return gfail(-1, "%s: null pointer argument", fn);
    if (nx <= 0 || ny <= 0 || nz <= 0 || n < 0 || !(cell > 0.0)) return gfail(-2, "%s: bad dims, count or cell", fn);
    if (grid_dtype != SDFR_F32 && grid_dtype != SDFR_U16)
        return gfail(-3, "%s: grid dtype must be f32 or u16 (got %d)", fn, grid_dtype);
    if (pos_dtype != SDFR_F32 && pos_dtype != SDFR_F64)
        return gfail(-3, "%s: position dtype must be f32 or f64 (got %d)", fn, pos_dtype);
    if (pos_stride < 3) return gfail(-2, "%s: position row stride below 3", fn);
    if (n > (int64_t)0x7fffffff * per_block) return gfail(-2, "%s: too many positions", fn);
    // GoalField.__init__ (goalfield.py:59-66): Python floats, compared in fp32
    *a = {grid, quant, nx, ny, nz, mins[0], mins[1], mins[2], cell,
          (float)(reach_max + 0.5 * cell), (float)(reach_max + 2.0 * cell)};
    return 0;
}

#define GOAL_LAUNCH(KERNEL, PER_BLOCK)                                                             \
    do {                                                                                           \
        const int blocks = (int)((n + (PER_BLOCK)-1) / (PER_BLOCK));                               \
        hipStream_t st = (hipStream_t)stream;                                                      \
        if (grid_dtype == SDFR_F32 && pos_dtype == SDFR_F64)                                       \
            KERNEL<SDFR_F32, SDFR_F64><<<blocks, 256, 0, st>>>(a, pos, pos_stride, n, out);        \
        else if (grid_dtype == SDFR_F32)                                                           \
            KERNEL<SDFR_F32, SDFR_F32><<<blocks, 256, 0, st>>>(a, pos, pos_stride, n, out);        \
        else if (pos_dtype == SDFR_F64)                                                            \
            KERNEL<SDFR_U16, SDFR_F64><<<blocks, 256, 0, st>>>(a, pos, pos_stride, n, out);        \
        else                                                                                       \
            KERNEL<SDFR_U16, SDFR_F32><<<blocks, 256, 0, st>>>(a, pos, pos_stride, n, out);        \
    } while (0)

SDFR_API int32_t sdfr_goal_sample(const void* grid, int32_t grid_dtype, float quant, int32_t nx,
                                  int32_t ny, int32_t nz, const double* mins, double cell,
                                  double reach_max, const void* pos, int32_t pos_dtype,
                                  int64_t pos_stride, int64_t n, float* out, void* stream) {
    FieldArgs a;
    const int32_t rc = field_args("sdfr_goal_sample", &a, grid, grid_dtype, quant, nx, ny, nz, mins, cell, reach_max,
                                  pos, pos_dtype, pos_stride, n, out, 256);
    if (rc != 0 || n == 0) return rc;
    GOAL_LAUNCH(goal_sample, 256);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return gfail(-4, "sdfr_goal_sample: launch failed: %s", hipGetErrorString(e));
    return 0;
}

SDFR_API int32_t sdfr_goal_yaw(const void* grid, int32_t grid_dtype, float quant, int32_t nx, int32_t ny, int32_t nz,
                               const double* mins, double cell, double reach_max, const void* pos, int32_t pos_dtype,
                               int64_t pos_stride, int64_t n, float* out, void* stream) {
    FieldArgs a;
    const int32_t rc = field_args("sdfr_goal_yaw", &a, grid, grid_dtype, quant, nx, ny, nz, mins, cell, reach_max, pos,
                                  pos_dtype, pos_stride, n, out, 64);
    if (rc != 0 || n == 0) return rc;
    GOAL_LAUNCH(goal_yaw, 64);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return gfail(-4, "sdfr_goal_yaw: launch failed: %s", hipGetErrorString(e));
    return 0;
}
#undef GOAL_LAUNCH

}  // extern "C"
