// edt.hip — exact Euclidean distance transform of a voxel occupancy grid on
// the GPU: the SDF bake of the reference's build_sdf (python/surfgym/vision.py
// :428-438), which pads the occupancy with one layer of solid and calls
//   scipy.ndimage.distance_transform_edt(occ == 0, sampling=cell)
// then crops the padding and stores f32 (f16 above 100 M voxels).
//
// Method: the squared distance transform is separable (Felzenszwalb &
// Huttenlocher, "Distance Transforms of Sampled Functions", 2012). Three
// passes:
//   x: one wave per row: each voxel's distance to the nearest solid in its
//      row (the padding makes x = -1 and x = nx solid), squared: g^2;
//   y: one thread per column: lower envelope of the parabolas
//      f(q) + (y - q)^2 over the column, with the padded rows q = -1 and
//      q = ny at f = 0;
//   z: the same along z, then d = sqrt(D * cell^2) in fp64, rounded once.
// All envelope arithmetic is exact integer arithmetic (squared distances in
// voxel units fit in int32, intersection comparisons are cross-multiplied in
// int64), so the squared distance of every voxel is exact. For a power-of-two
// cell (every cell pick_cell chooses, vision.py:283-298) scipy's float64
// sum of per-axis squares equals cell^2 * D exactly, so the result is
// bit-identical to the reference's bake.
//
// The passes have two implementations with identical results: tiles of lines
// staged in LDS, 16-bit or 32-bit squares (edt_pack, edt_tile), wherever the y
// and z lines fit; and, for longer lines, the walk above (edt_rows, edt_cols,
// edt_slabs; one thread per y or z line).
//
// Scratch: two int32 planes of the grid and one uint64 envelope stack per
// line (~16 bytes per voxel, sdfr_edt_workspace_bytes); the tiles use 2.25 bytes
// per voxel of it in long rows of up to 509 planes, 12 at most (rows of one
// voxel).

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <string.h>

#include <type_traits>

#include "../../include/sdfr.h"

namespace {

thread_local char e_err[256];

__attribute__((format(printf, 2, 3))) int32_t efail(int32_t code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(e_err, sizeof e_err, fmt, ap);
    va_end(ap);
    return code;
}

// fp64 -> fp16, rounded once to nearest even (numpy's astype(float16)):
// round to fp32 toward zero and set the sticky bit if anything was dropped
// (round-to-odd keeps enough bits for the second rounding to be exact), then
// round that to fp16.
__device__ __forceinline__ __half f64_to_f16_rne(double x) {
    float t = __double2float_rz(x);
    if ((double)t != x) t = __uint_as_float(__float_as_uint(t) | 1u);
    return __float2half_rn(t);
}

// Pass x: per row, distance to the nearest solid (pads at -1 and nx), squared.
// One wave per row; lane l owns the run x in [l*C, (l+1)*C), C = ceil(nx/64).
// The nearest solid at or left of x is the last solid in the lane's run up to
// x, else the last solid of any lower lane (a prefix max over the wave), else
// the pad at -1; the right side mirrors it with a suffix min and the pad at nx.
__global__ __launch_bounds__(256) void edt_rows(const uint8_t* __restrict__ occ, int32_t* __restrict__ g,
                                                int nx, int64_t rows) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;   // uniform per wave
    const int lane = threadIdx.x & 63;
    const int C = (nx + 63) >> 6;
    const int x0 = min(lane * C, nx), x1 = min(x0 + C, nx);
    const uint8_t* o = occ + row * nx;
    int32_t* out = g + row * nx;
    int first = nx, last = -1;   // solids in this lane's run
    for (int x = x0; x < x1; ++x)
        if (o[x]) {
            first = min(first, x);
            last = x;
        }
    // inclusive scans over the wave: max of `last` up from lane 0, min of
    // `first` down from lane 63
    int lmax = last, rmin = first;
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(lmax, off);
        const int dn = __shfl_down(rmin, off);
        if (lane >= off) lmax = max(lmax, up);
        if (lane + off < 64) rmin = min(rmin, dn);
    }
    int left = __shfl_up(lmax, 1);     // last solid below this lane's run
    int right = __shfl_down(rmin, 1);  // first solid above it
    if (lane == 0) left = -1;
    if (lane == 63) right = nx;
    for (int x = x0; x < x1; ++x) {
        if (o[x]) left = x;
        out[x] = x - left;
    }
    for (int x = x1 - 1; x >= x0; --x) {
        if (o[x]) right = x;
        const int32_t m = min(out[x], right - x);
        out[x] = m * m;
    }
}

// One column of the lower-envelope pass. The column has n real samples at
// stride `stride` from `f`, plus pad samples q = -1 and q = n with value 0.
// A parabola rooted at p is kept as (p, H) with H = f(p) + p^2, so the
// intersection of the parabolas rooted at a < b is
//   s(a, b) = (H_b - H_a) / (2 (b - a)),
// compared as cross-multiplied int64 fractions (exact). The envelope stack
// lives in `v` (stride `vstride`), one uint64 per vertex: H << 16 | (p + 1)
// (H < 2^32 and p + 1 < 2^16 under sdfr_edt's size checks); its top two
// vertices are kept in registers, so popping one costs a single dependent
// load, and the next sample is fetched while the current one is placed.
__device__ __forceinline__ int64_t fval(const int32_t* f, int64_t stride, int n, int q) {
    return (q < 0 || q >= n) ? 0 : (int64_t)f[(int64_t)q * stride];
}

struct Vtx {
    int p;       // root
    int64_t h;   // f(p) + p^2
};

__device__ __forceinline__ uint64_t pack_vtx(Vtx a) {
    return ((uint64_t)a.h << 16) | (uint64_t)(a.p + 1);
}

__device__ __forceinline__ Vtx unpack_vtx(uint64_t w) {
    return Vtx{(int)(w & 0xffffu) - 1, (int64_t)(w >> 16)};
}

__device__ __forceinline__ void envelope_line(const int32_t* __restrict__ f, int64_t stride, int n,
                                              uint64_t* __restrict__ v, int64_t vstride,
                                              int32_t* __restrict__ out, int64_t ostride,
                                              bool last, float* __restrict__ fout,
                                              __half* __restrict__ hout, double cell2) {
    // build the envelope over q = -1 .. n
    int k = 0;                          // index of the top vertex
    Vtx top{-1, 1};                     // the pad at q = -1: f = 0
    Vtx second{0, 0};                   // valid while k >= 1
    v[0] = pack_vtx(top);
    // the samples come in chunks of kChunk, the next chunk's loads in flight
    // while this one is placed (they do not depend on the envelope)
    constexpr int kChunk = 16;
    int64_t fc[kChunk], fn[kChunk];
#pragma unroll
    for (int i = 0; i < kChunk; ++i) fc[i] = fval(f, stride, n, i);
    for (int q0 = 0; q0 <= n; q0 += kChunk) {
#pragma unroll
        for (int i = 0; i < kChunk; ++i) fn[i] = fval(f, stride, n, q0 + kChunk + i);
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
            const int q = q0 + i;
            if (q > n) break;
            const int64_t hq = fc[i] + (int64_t)q * q;
            while (k > 0) {
                // pop the top while q's parabola takes over at or before the
                // point where the top took over from the vertex below it:
                // s(top, q) <= s(second, top)
                const int64_t s_num = hq - top.h, s_den = 2 * (int64_t)(q - top.p);
                const int64_t z_num = top.h - second.h, z_den = 2 * (int64_t)(top.p - second.p);
                if (s_num * z_den > z_num * s_den) break;
                --k;
                top = second;
                if (k > 0) second = unpack_vtx(v[(int64_t)(k - 1) * vstride]);
            }
            ++k;
            second = top;
            top = Vtx{q, hq};
            v[(int64_t)k * vstride] = pack_vtx(top);
        }
#pragma unroll
        for (int i = 0; i < kChunk; ++i) fc[i] = fn[i];
    }
    // read the envelope at the real samples; vertices j .. j+3 in registers
    // (w[0] current, w[1] next), the later ones loaded ahead of their use
    int j = 0;
    uint64_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = i <= k ? v[(int64_t)i * vstride] : 0;
    Vtx cur = unpack_vtx(w[0]);
    for (int q = 0; q < n; ++q) {
        while (j < k) {
            // advance while the next vertex takes over before q: s(cur, nxt) < q
            const Vtx nxt = unpack_vtx(w[1]);
            const int64_t z_num = nxt.h - cur.h, z_den = 2 * (int64_t)(nxt.p - cur.p);
            if (z_num >= (int64_t)q * z_den) break;
            ++j;
            cur = nxt;
            w[1] = w[2];
            w[2] = w[3];
            w[3] = j + 3 <= k ? v[(int64_t)(j + 3) * vstride] : 0;
        }
        const int64_t d = (int64_t)(q - cur.p) * (q - cur.p) + (cur.h - (int64_t)cur.p * cur.p);
        if (!last) {
            out[(int64_t)q * ostride] = (int32_t)d;
        } else {
            const double dist = sqrt((double)d * cell2);
            if (fout) fout[(int64_t)q * ostride] = (float)dist;
            else hout[(int64_t)q * ostride] = f64_to_f16_rne(dist);
        }
    }
}

// Pass y: one thread per (z, x) column of a [nz][ny][nx] plane array.
__global__ __launch_bounds__(256) void edt_cols(const int32_t* __restrict__ f, int32_t* __restrict__ out,
                                                uint64_t* __restrict__ v, int nx, int ny, int nz) {
    const int64_t line = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t lines = (int64_t)nz * nx;
    if (line >= lines) return;
    const int z = (int)(line / nx), x = (int)(line - (int64_t)z * nx);
    const int64_t base = (int64_t)z * ny * nx + x;
    // envelope stack: entry j of this line at v[j*lines + line] (coalesced)
    envelope_line(f + base, nx, ny, v + line, lines, out + base, nx, false, nullptr, nullptr, 0.0);
}

// Pass z: one thread per (y, x) line; writes the distances.
__global__ __launch_bounds__(256) void edt_slabs(const int32_t* __restrict__ f, uint64_t* __restrict__ v,
                                                 float* __restrict__ fout, __half* __restrict__ hout,
                                                 int nx, int ny, int nz, double cell2) {
    const int64_t line = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t lines = (int64_t)ny * nx;
    if (line >= lines) return;
    const int64_t plane = (int64_t)ny * nx;
    envelope_line(f + line, plane, nz, v + line, lines, nullptr, plane, true,
                  fout ? fout + line : nullptr, hout ? hout + line : nullptr, cell2);
}

// ------------------------------------------------------------- tiled passes --
// The transform in three kernels that move 5.5 bytes a voxel and the output
// between them (a byte of occupancy, a quarter byte of packed bits each way,
// 16-bit squares each way). A pass searches, for every output q of a line,
// D(q) = min over p of f(p) + (q - p)^2 over whole lines staged in LDS.
//
//   * Only what can still win is kept. The solid layer above and below the
//     grid bounds every distance along z by min(z + 1, nz - z), and a value
//     f(p) at plane p can only take part in one of them if it is below
//         max over q of min(q + 1, nz - q)^2 - (q - p)^2 = (p + 1)(nz - p):
//     the first bound grows with q, the second falls, they meet at
//     2q = nz - 1. So values of the x and y passes are clamped there (z_cap)
//     without changing a result, which also bounds the y search by
//     sqrt(z_cap); for nz <= 509 the squares fit 16 bits (two voxels a
//     register, v_pk_add_u16 saturating and v_pk_min_u16) and the distances
//     along x a byte.
//   * A thread takes BLK consecutive outputs of a line (two lines when
//     packed) in registers and reads each candidate once for all of them.
//   * Candidates come in chunks of BLK rows, nearest first, on both sides,
//     until even a zero in the next chunk could not win (its nearest row is
//     BLK(c - 1) + 1 away); a chunk whose smallest value (kept per chunk and
//     line) cannot win at that distance either is skipped. Neighbouring lines
//     agree about both, so on the scenes measured a wave searches ~4 of a
//     line's 128 chunks.
//
// What bounds it: at 1024x1024x256 voxels (125 + 755 + 622 us; 3049 + 4881 +
// 3207 for a wave per row and a walk per line) vector issue, 60, 69 and 85% of
// the cycles in the packing, y and z passes, and in the y pass the waits for its
// tiles besides. At 256x256x128 (6 + 31 + 26 us; 36 + 98 + 62 for a wave per row
// and a search per output) all tiles are in flight at once, vector issue is 14,
// 38 and 41%, and a wave spends 40% of its time waiting for its tile and its
// group and 36% for its turn at the SIMD; LDS is busy 4% of the time, without a
// bank conflict. The bytes alone take 410 and 16 us at a copy's 4.9 TB/s. 8
// outputs a thread beat 16 (40 + 32, 887 + 831 us) as they leave twice the waves
// in flight (2 in small grids: small_grid); tiles 32 words wide beat 64, of which
// fewer fit a CU (33 + 27, 1077 + 785 us); 1024 threads beat 512 in the y pass,
// whose tiles fill the LDS (749 against 930 us), and lose in the z pass (741
// against 622).
//
// The walk per line that the tiles replaced (a search per output for few lines)
// was timed against them on grids of 64x64x300 to 1024^3 voxels, empty, with a
// floor and boxes, and with one voxel in 10^5 and in 100 solid: the tiles win on
// all, by least on empty cubes in 32 bits (640^3 9.1 -> 4.5 ms, 1024^3 47.7 ->
// 23.9), and also with one narrow tile a CU (z lines of 4000 voxels: 300x300x4000
// 13.7 -> 4.8 ms; y lines of 8000: 200x8000x300 21 -> 3.4 ms), so only the lines
// that do not fit walk.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kBlk = 8;       // outputs a thread takes and rows a chunk holds, ...
constexpr int kSmallBlk = 2;  // ... and in small grids (small_grid)
constexpr int kThreadsY = 1024, kThreadsZ = 512;

template <typename V> struct Word;
template <> struct Word<u16x2> {   // two voxels, 16-bit squares
    typedef uint16_t Plane;
    static constexpr int kVox = 2;
    static constexpr uint32_t kMax = 0xffffu;
    static __device__ __forceinline__ u16x2 splat(uint32_t v) {
        const unsigned short h = (unsigned short)v;
        return u16x2{h, h};
    }
    static __device__ __forceinline__ u16x2 add(u16x2 a, u16x2 b) { return __builtin_elementwise_add_sat(a, b); }
    static __device__ __forceinline__ bool any_less(u16x2 a, u16x2 b) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(b, a)) != 0u;
    }
    static __device__ __forceinline__ uint32_t get(u16x2 v, int i) { return i ? v.y : v.x; }
};
template <> struct Word<uint32_t> {   // one voxel
    typedef uint32_t Plane;
    static constexpr int kVox = 1;
    static constexpr uint32_t kMax = 0x3fffffffu;   // kMax + any (q - p)^2 stays below 2^32
    static __device__ __forceinline__ uint32_t splat(uint32_t v) { return v; }
    static __device__ __forceinline__ uint32_t add(uint32_t a, uint32_t b) { return a + b; }
    static __device__ __forceinline__ bool any_less(uint32_t a, uint32_t b) { return a < b; }
    static __device__ __forceinline__ uint32_t get(uint32_t v, int) { return v; }
};

// What a tile holds per word in LDS: the squares, or in the packed y pass the
// two distances along x in a byte each, squared when they are read.
template <typename V, bool Z> struct Cell {
    typedef V T;
    static __device__ __forceinline__ V open(T c) { return c; }
    static __device__ __forceinline__ T shut(V v) { return v; }
    static __device__ __forceinline__ V value(V v) { return v; }
    static __device__ __forceinline__ V far() { return Word<V>::splat(Word<V>::kMax); }
};
template <> struct Cell<u16x2, false> {
    typedef uint16_t T;
    static __device__ __forceinline__ u16x2 open(T c) {
        return __builtin_bit_cast(u16x2, (uint32_t)__builtin_amdgcn_perm(0u, c, 0x0c010c00u));
    }
    static __device__ __forceinline__ T shut(u16x2 v) { return (T)(v.x | (v.y << 8)); }
    static __device__ __forceinline__ u16x2 value(u16x2 v) { return v * v; }
    static __device__ __forceinline__ u16x2 far() { return Word<u16x2>::splat(255u); }
};

// Block b runs on XCD b % 8; give each XCD a contiguous run of tiles, so that
// tiles beside each other along x, which share 128-byte lines, share an L2.
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t n) {
    const int64_t q = n >> 3, rem = n & 7, x = b & 7;
    return x * q + (x < rem ? x : rem) + (b >> 3);
}

// Pass x: the occupancy as bits. Per 32 voxels of a row (voxels past its end
// count as solid: they are the padding): the bits, the distance from the
// first voxel back to the last solid before it (low 16 bits) and from the
// last voxel to the first solid after it (high 16). A quarter byte a voxel,
// from which the y pass forms any voxel's distance with two bit scans. Laid
// out [nz][words][ny], so that a tile's rows are consecutive.
// R rows of a block are packed into LDS, then each (row, word) looks outward
// for the nearest word that holds a solid.
__global__ __launch_bounds__(256) void edt_pack(const uint8_t* __restrict__ occ, uint2* __restrict__ bits,
                                                int nx, int ny, int64_t rows, int words, int R, int wide) {
    extern __shared__ uint32_t s[];
    const int64_t row0 = (int64_t)blockIdx.x * R;
    const int ls = words + 1;                 // odd-even row stride against bank conflicts
    uint16_t* half = (uint16_t*)s;
    const int halves = 2 * words;
    for (int i = threadIdx.x; i < R * halves; i += 256) {
        const int r = i / halves, h = i - r * halves;
        const int x0 = h * 16;
        uint32_t b = 0xffffu;
        if (row0 + r < rows && x0 < nx) {
            const uint8_t* o = occ + (row0 + r) * nx + x0;
            if (wide) {   // nx a multiple of 16 and occ 16-byte aligned
                const uint4 v = *(const uint4*)o;
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
                b = 0u;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    // bit 7 of each non-zero byte, gathered into 4 bits
                    const uint32_t nz = (((w[k] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[k]) & 0x80808080u;
                    b |= (((nz >> 7) * 0x01020408u) >> 24) << (4 * k);
                }
            } else {
                b = 0u;
#pragma unroll
                for (int k = 0; k < 16; ++k)
                    b |= (x0 + k >= nx || o[k] != 0 ? 1u : 0u) << k;
            }
        }
        half[r * 2 * ls + h] = (uint16_t)b;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < R * words; i += 256) {
        const int w = i / R, r = i - w * R;
        if (row0 + r >= rows) continue;
        const uint32_t* line = s + r * ls;
        int k = w - 1;
        while (k >= 0 && line[k] == 0u) --k;
        const int left = k < 0 ? 32 * w + 1 : 32 * w - (32 * k + 31 - __builtin_clz(line[k]));
        k = w + 1;
        while (k < words && line[k] == 0u) ++k;
        // past the last word everything is padding; so is its tail
        const int right = k >= words ? 32 * words - (32 * w + 31) : 32 * k + __builtin_ctz(line[k]) - (32 * w + 31);
        const int64_t row = row0 + r, z = row / ny, y = row - z * ny;
        bits[(z * words + w) * ny + y] = make_uint2(line[w], (uint32_t)left | ((uint32_t)right << 16));
    }
}

// Zeros above the top set bit / below the bottom one; no set bit: 2^32 - 1.
__device__ __forceinline__ uint32_t top_zeros(uint32_t v) { return v ? (uint32_t)__builtin_clz(v) : 0xffffffffu; }
__device__ __forceinline__ uint32_t low_zeros(uint32_t v) { return v ? (uint32_t)__builtin_ctz(v) : 0xffffffffu; }

// Distance along x of voxel i (0..31) of a packed word to the nearest solid.
__device__ __forceinline__ uint32_t row_distance(uint2 b, int i) {
    const uint32_t left = (uint32_t)i + (b.y & 0xffffu), right = (uint32_t)(31 - i) + (b.y >> 16);
    return min(min(top_zeros(b.x << (31 - i)), low_zeros(b.x >> i)), min(left, right));
}

// sqrt(x) rounded to nearest, for x >= 2^-60 or 0 of the normal range: the
// hardware root is within one ulp, and of the three candidates the one whose
// products with the root bracket x is the rounded one (Markstein's test).
// For an x that fp32 holds exactly this is the fp64 root rounded to fp32
// (double rounding is harmless for a root: 53 >= 2*24 + 2 bits).
__device__ __forceinline__ float sqrt_rn(float x) {
    float r = __builtin_amdgcn_sqrtf(x);
    const float lo = __uint_as_float(__float_as_uint(r) - 1u), hi = __uint_as_float(__float_as_uint(r) + 1u);
    const float below = __builtin_fmaf(-lo, r, x), above = __builtin_fmaf(-hi, r, x);
    r = below <= 0.0f ? lo : r;
    return above > 0.0f ? hi : r;
}

// The same rounded once to fp16 (results of at least 2^-14, or 0): the root
// lies in the fp16 interval of the hardware's, or an ulp beside one of its
// ends, so comparing x with the square of the interval's midpoint rounds it.
__device__ __forceinline__ __half sqrt_rn_f16(float x) {
    const uint32_t lo = __float_as_uint(__builtin_amdgcn_sqrtf(x)) & ~0x1fffu;
    const float mid = __uint_as_float(lo | 0x1000u);
    const float rem = __builtin_fmaf(-mid, mid, x);
    const bool up = rem > 0.0f || (rem == 0.0f && (lo & 0x2000u) != 0u);
    return __float2half_rn(__uint_as_float(up ? lo + 0x2000u : lo));
}

struct PassArgs {
    const uint2* bits;     // y pass: packed occupancy
    void* plane;           // squared distances over x and y, pitch voxels a row
    int pitch;
    void* out;             // y pass: the plane; z pass: the distances
    int nx, ny, nz, words;
    int n, blks;           // line length and its blocks of BLK rows
    int tiles;             // tiles along x
    int64_t blocks;
    double cell2;
    float cell2f;          // cell2 in fp32 (where D * cell2 is exact there)
    int wide;              // z pass: two voxels a store (a row holds a whole number of pairs)
};

// Row of a tile in LDS: a row's gap after each block of rows, so that the
// blocks a wave works on lie on different banks.
template <int TW, int BLK>
__device__ __forceinline__ int tile_row(int row) {
    return (row + row / BLK) * TW;
}

// What a pass writes: the plane of squares (y pass), or the distances.
enum { kPlane, kF32, kF16 };

// The distance of a squared one: fp32 or fp16, rounded once from sqrt(d * cell2).
template <typename O, bool EXACT>
__device__ __forceinline__ O distance(const PassArgs& a, uint32_t d) {
    if constexpr (std::is_same<O, float>::value) {
        if constexpr (EXACT) return sqrt_rn((float)d * a.cell2f);
        else return (float)sqrt((double)d * a.cell2);
    } else {
        if constexpr (EXACT) return sqrt_rn_f16((float)d * a.cell2f);
        else return f64_to_f16_rne(sqrt((double)d * a.cell2));
    }
}

template <typename V, typename O, bool EXACT>
__device__ __forceinline__ void put_distances(const PassArgs& a, O* o, V v, int x) {
    const O d0 = distance<O, EXACT>(a, Word<V>::get(v, 0));
    if constexpr (Word<V>::kVox == 2) {
        const O d1 = distance<O, EXACT>(a, Word<V>::get(v, 1));
        struct alignas(2 * sizeof(O)) Two { O a, b; };
        if (a.wide) *(Two*)o = Two{d0, d1};
        else {
            o[0] = d0;
            if (x + 1 < a.nx) o[1] = d1;
        }
    } else {
        o[0] = d0;
    }
}

template <typename V, int TW, int OUT, bool EXACT, int BLK>
__global__ __launch_bounds__(OUT == kPlane ? kThreadsY : kThreadsZ) void edt_tile(PassArgs a) {
    constexpr bool Z = OUT != kPlane;
    using W = Word<V>;
    using P = typename W::Plane;
    using C = Cell<V, Z>;
    using T = typename C::T;
    extern __shared__ uint32_t smem[];
    T* s = (T*)smem;                                                  // the tile's lines
    T* cmin = s + (size_t)tile_row<TW, BLK>(a.blks * BLK);                // smallest of each chunk
    const int64_t tile = xcd_tile(blockIdx.x, a.blocks);
    const int outer = (int)(tile / a.tiles);             // z (y pass) or y (z pass)
    const int xt = (int)(tile - (int64_t)outer * a.tiles) * TW * W::kVox;
    const int n = a.n;

    // a thread keeps its column: the workgroup is a multiple of TW wide
    const int col = threadIdx.x % TW, x = xt + col * W::kVox;
    const int row0 = threadIdx.x / TW, rows = blockDim.x / TW;
    if constexpr (Z) {
        const P* p = (const P*)a.plane + (int64_t)outer * a.pitch + x;
        const int64_t step = (int64_t)a.ny * a.pitch;
        for (int row = row0; row < a.blks * BLK; row += rows)
            s[tile_row<TW, BLK>(row) + col] = row < n && x < a.nx ? C::shut(*(const V*)(p + row * step)) : C::shut(C::far());
    } else {
        const uint2* p = a.bits + ((int64_t)outer * a.words + (x >> 5)) * n;
        const int i = x & 31;
        for (int row = row0; row < a.blks * BLK; row += rows) {
            V v = C::far();
            if (row < n && x < a.nx) {
                const uint2 b = p[row];
                const uint32_t g0 = row_distance(b, i);
                if constexpr (W::kVox == 2) {
                    const uint32_t g1 = row_distance(b, i + 1);
                    v = u16x2{(unsigned short)min(g0, 255u), (unsigned short)min(g1, 255u)};
                } else {
                    v = g0 * g0;
                }
            }
            s[tile_row<TW, BLK>(row) + col] = C::shut(v);
        }
    }
    __syncthreads();
    for (int k = row0; k < a.blks; k += rows) {
        const T* p = s + tile_row<TW, BLK>(k * BLK) + col;
        V m = C::open(p[0]);
#pragma unroll
        for (int r = 1; r < BLK; ++r) m = __builtin_elementwise_min(m, C::open(p[r * TW]));
        cmin[k * TW + col] = C::shut(m);
    }
    __syncthreads();
    if (x >= a.nx) return;
    const uint32_t cap = Z ? W::kMax : min((uint32_t)(outer + 1) * (uint32_t)(a.nz - outer), W::kMax);   // z_cap
    for (int blk = row0; blk < a.blks; blk += rows) {
        const int q0 = blk * BLK;
        const T* own = s + tile_row<TW, BLK>(q0) + col;
        V best[BLK];
        V most = W::splat(0u);
#pragma unroll
        for (int r = 0; r < BLK; ++r) {
            // the value above, and the solid rows at -1 and n; rows past the
            // end take part in nothing
            const int e = min(q0 + r + 1, n - q0 - r);
            const uint32_t pad = e > 0 ? min((uint32_t)(e * e), cap) : 0u;
            best[r] = __builtin_elementwise_min(C::value(C::open(own[r * TW])), W::splat(pad));
            most = __builtin_elementwise_max(most, best[r]);
        }
        // the chunk of rows at p, row j at distance d(j, r) from output r
        auto take = [&](const T* p, auto square) {
#pragma unroll
            for (int j = 0; j < BLK; ++j) {
                const V v = C::value(C::open(p[j * TW]));
#pragma unroll
                for (int r = 0; r < BLK; ++r)
                    best[r] = __builtin_elementwise_min(best[r], W::add(v, square(j, r)));
            }
            most = best[0];
#pragma unroll
            for (int r = 1; r < BLK; ++r) most = __builtin_elementwise_max(most, best[r]);
        };
        if (W::any_less(C::value(C::open(cmin[blk * TW + col])), most))
            take(own, [](int j, int r) { return W::splat((uint32_t)((j - r) * (j - r))); });
        for (int c = 1;; ++c) {
            const uint32_t near = (uint32_t)(BLK * (c - 1) + 1);   // of the chunk's nearest row
            const V near2 = W::splat(min(near * near, W::kMax));
            const bool go = W::any_less(near2, most);
            if (!__any(go)) break;
            const int up = blk + c, down = blk - c;
            const bool has_up = up < a.blks, has_down = down >= 0;
            if (!__any(has_up || has_down)) break;
            // row j is near + j beyond the last output or before the first
            V sq[2 * BLK - 1];
#pragma unroll
            for (int k = 0; k < 2 * BLK - 1; ++k)
                sq[k] = W::splat(min((near + (uint32_t)k) * (near + (uint32_t)k), W::kMax));
            if (go && has_up && W::any_less(W::add(C::value(C::open(cmin[up * TW + col])), near2), most))
                take(s + tile_row<TW, BLK>(up * BLK) + col, [&](int j, int r) { return sq[j + BLK - 1 - r]; });
            if (go && has_down && W::any_less(W::add(C::value(C::open(cmin[down * TW + col])), near2), most))
                take(s + tile_row<TW, BLK>(down * BLK) + col, [&](int j, int r) { return sq[BLK - 1 - j + r]; });
        }
        const int64_t step = Z ? (int64_t)a.ny * a.nx : a.pitch;
        const int64_t first = Z ? ((int64_t)q0 * a.ny + outer) * a.nx + x : ((int64_t)outer * n + q0) * a.pitch + x;
        using O = typename std::conditional<OUT == kPlane, P, typename std::conditional<OUT == kF32, float, __half>::type>::type;
        O* o = (O*)a.out + first;
#pragma unroll
        for (int r = 0; r < BLK; ++r) {
            if (q0 + r < n) {
                if constexpr (!Z) *(V*)(o + r * step) = best[r];
                else put_distances<V, O, EXACT>(a, o + r * step, best[r], x);
            }
        }
    }
}

// Whether a grid has too few rows, and too short searches (the z bound), to
// fill the GPU with kBlk outputs a thread. What bounds its passes is one
// thread's chain: its loads in turn, and searches unrolled into more code than
// they run. kSmallBlk shortens both, and edt_pack takes fewer rows a block.
// The three launches in a graph, us, 1% of the voxels solid (none in the last
// three rows), with a wave a row and a search per output / kBlk / kSmallBlk and
// the short blocks of edt_pack:
//   40x40x16 voxels 11.3 / 15.9 / 11.7     200x40x16 13.5 / 19.5 / 13.1
//   300x60x16       17.0 / 21.2 / 13.7     900x40x16 26.3 / 25.6 / 15.3
//   64x64x64        28.7 / 18.3 / 18.4 (the last on this side of both lines)
//   40x40x128       39.5 / 16.4 / 24.5
//   300x300x16       117 / 25.7 / 28.3
bool small_grid(int nx, int ny, int nz) {
    const int64_t rows = (int64_t)ny * nz;
    return rows <= 4096 && rows * nx * nz <= 1 << 24;
}

// Words a tile is wide for lines of n, and its LDS bytes; 0 where even the
// narrowest does not fit the workgroup's LDS. Rows `across` words long get no
// wider tile than covers them: its other lanes would work on padding (1x1500x40
// voxels 48 us 32 words wide, 21 us 8 wide; 16x200x600 46 and 30).
int tile_words(int n, int across, int blk, int cell_bytes, int64_t lds_limit, size_t* lds) {
    const int64_t blks = (n + blk - 1) / blk;
    for (int tw : {32, 16, 8}) {
        if (tw > 8 && tw / 2 >= across) continue;
        const int64_t bytes = blks * (blk + 2) * tw * cell_bytes;   // rows, gap and minimum
        if (bytes <= lds_limit) {
            *lds = (size_t)bytes;
            return tw;
        }
    }
    return 0;
}

// A pass's tiles: `blk` outputs a thread, `tw` words wide, `lds` bytes of the
// device's `limit`.
struct TilePlan {
    int blk, tw, limit;
    size_t lds;
};

template <typename V, int OUT, bool EXACT, int BLK>
hipError_t launch_tile(PassArgs a, const TilePlan& t, int outer, hipStream_t st) {
    const int tw = t.tw;
    a.blks = (a.n + BLK - 1) / BLK;
    const int vox = tw * Word<V>::kVox;
    a.tiles = (a.nx + vox - 1) / vox;
    a.blocks = (int64_t)a.tiles * outer;
    auto* k = tw == 32   ? edt_tile<V, 32, OUT, EXACT, BLK>
              : tw == 16 ? edt_tile<V, 16, OUT, EXACT, BLK>
                         : edt_tile<V, 8, OUT, EXACT, BLK>;
    if (t.lds > (64 << 10)) {
        // the attribute belongs to the process: every call sets the device's
        // limit, not its own size, so that no thread's launch meets a smaller
        // size that another thread has set for its grid
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, t.limit);
        if (e != hipSuccess) return e;
    }
    const int items = a.blks * tw;   // one BLK-output search each
    const int most = OUT == kPlane ? kThreadsY : kThreadsZ;
    const int threads = items >= most ? most : (items + 63) & ~63;
    k<<<(unsigned)a.blocks, threads, t.lds, st>>>(a);
    return hipGetLastError();
}

template <typename V, int OUT, bool EXACT>
hipError_t launch_tile(const PassArgs& a, const TilePlan& t, int outer, hipStream_t st) {
    return t.blk == kBlk ? launch_tile<V, OUT, EXACT, kBlk>(a, t, outer, st)
                         : launch_tile<V, OUT, EXACT, kSmallBlk>(a, t, outer, st);
}

template <typename V>
hipError_t launch_z(const PassArgs& a, bool f32, bool exact, const TilePlan& t, hipStream_t st) {
    if (f32) return exact ? launch_tile<V, kF32, true>(a, t, a.ny, st) : launch_tile<V, kF32, false>(a, t, a.ny, st);
    return exact ? launch_tile<V, kF16, true>(a, t, a.ny, st) : launch_tile<V, kF16, false>(a, t, a.ny, st);
}

// Bytes hold every distance along x that can matter (255^2 >= z_cap), and 16
// bits every square, up to this nz: floor((nz + 1)^2 / 4) <= 65025.
constexpr int kPackedMaxNz = 509;

// Whether D * cell2 is exact in fp32 for every squared distance D a grid can
// hold (the padding bounds D by ((n + 1) / 2)^2 along the shortest axis).
bool exact_in_f32(double cell2, int nx, int ny, int nz) {
    const int64_t n = nx < ny ? (nx < nz ? nx : nz) : (ny < nz ? ny : nz);
    const int64_t most = ((n + 1) / 2) * ((n + 1) / 2);
    int e = 0;
    double m = frexp(cell2, &e);
    int bits = 0;
    while (bits < 54 && m != floor(m)) {
        m *= 2.0;
        ++bits;
    }
    return (double)most * m < 16777216.0 && cell2 >= 0x1p-28 && cell2 * (double)most < 0x1p100;
}

// Two int32 planes of the grid, then (8-byte aligned) the uint64 envelope
// stacks of the longer of the y and z passes.
int64_t edt_env_offset(int nx, int ny, int nz) {
    const int64_t vox = (int64_t)nx * ny * nz;
    return (2 * vox * (int64_t)sizeof(int32_t) + 7) & ~(int64_t)7;
}

int64_t edt_scratch_bytes(int nx, int ny, int nz) {
    const int64_t lines_y = (int64_t)nz * nx, lines_z = (int64_t)ny * nx;
    const int64_t venv = lines_y * (ny + 2) > lines_z * (nz + 2) ? lines_y * (ny + 2)
                                                                 : lines_z * (nz + 2);
    return edt_env_offset(nx, ny, nz) + venv * (int64_t)sizeof(uint64_t);
}

}  // namespace

extern "C" {

SDFR_API int64_t sdfr_edt_workspace_bytes(int32_t nx, int32_t ny, int32_t nz) {
    if (nx <= 0 || ny <= 0 || nz <= 0) return -2;
    return edt_scratch_bytes(nx, ny, nz);
}

SDFR_API const char* sdfr_edt_last_error(void) { return e_err; }

SDFR_API int32_t sdfr_edt(const uint8_t* occ, int32_t nx, int32_t ny, int32_t nz, float cell,
                          void* out, int32_t out_dtype, void* workspace, int64_t workspace_size,
                          void* stream) {
    e_err[0] = '\0';
    if (!occ || !out || !workspace) return efail(-1, "sdfr_edt: null pointer argument");
    if (nx <= 0 || ny <= 0 || nz <= 0)
        return efail(-2, "sdfr_edt: grid dims must be positive (got %d x %d x %d)", nx, ny, nz);
    if ((int64_t)nx + 2 > 46340 || (int64_t)ny + 2 > 46340 || (int64_t)nz + 2 > 46340)
        return efail(-2, "sdfr_edt: an axis longer than 46338 voxels overflows int32 distances");
    if ((int64_t)(nx + 2) * (nx + 2) + (int64_t)(ny + 2) * (ny + 2) + (int64_t)(nz + 2) * (nz + 2) >
        0x7fffffffLL)
        return efail(-2, "sdfr_edt: squared diagonal overflows int32");
    if (!(cell > 0.0f) || !isfinite(cell)) return efail(-2, "sdfr_edt: cell must be positive");
    if (out_dtype != SDFR_F32 && out_dtype != SDFR_F16)
        return efail(-3, "sdfr_edt: output dtype must be f32 or f16 (got %d)", out_dtype);
    const int64_t need = edt_scratch_bytes(nx, ny, nz);
    if (workspace_size < need)
        return efail(-2, "sdfr_edt: workspace of %lld bytes needed (got %lld)", (long long)need,
                     (long long)workspace_size);
    if (((uintptr_t)workspace & 7u) != 0) return efail(-2, "sdfr_edt: workspace must be 8-byte aligned");
    const int64_t vox = (int64_t)nx * ny * nz;
    hipStream_t st = (hipStream_t)stream;
    const double cell2 = (double)cell * (double)cell;
    const int64_t rows = (int64_t)nz * ny, cols = (int64_t)nz * nx, lines = (int64_t)ny * nx;
    float* fout = out_dtype == SDFR_F32 ? (float*)out : nullptr;
    __half* hout = out_dtype == SDFR_F16 ? (__half*)out : nullptr;
    int dev = 0, lds_limit = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds_limit, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        lds_limit = 64 << 10;
    const bool packed = nz <= kPackedMaxNz;
    const bool small = small_grid(nx, ny, nz);
    TilePlan ty, tz;
    ty.limit = tz.limit = lds_limit;
    const int across = packed ? (nx + 1) / 2 : nx;
    for (int blk : {kSmallBlk, kBlk}) {   // (1.6 times the LDS: a line that does not fit so may with kBlk)
        if (blk == kSmallBlk && !small) continue;
        ty.blk = tz.blk = blk;
        ty.tw = tile_words(ny, across, blk, packed ? 2 : 4, lds_limit, &ty.lds);
        tz.tw = tile_words(nz, across, blk, 4, lds_limit, &tz.lds);
        if (ty.tw && tz.tw) break;
    }
    if (ty.tw && tz.tw) {
        // the bits, then the plane of squares (edt_scratch_bytes holds both)
        PassArgs p;
        memset(&p, 0, sizeof p);
        p.words = (nx + 31) / 32;
        p.bits = (const uint2*)workspace;
        p.plane = (char*)workspace + rows * p.words * (int64_t)sizeof(uint2);
        p.pitch = packed ? (nx + 1) & ~1 : nx;
        p.nx = nx;
        p.ny = ny;
        p.nz = nz;
        p.cell2 = cell2;
        p.cell2f = (float)cell2;
        const bool exact = exact_in_f32(cell2, nx, ny, nz);
        p.wide = nx % 2 == 0 && ((uintptr_t)out & (fout ? 7u : 3u)) == 0;
        int R = (small ? 128 : 512) / p.words;   // 128: a half word a thread, in one round
        R = R < 1 ? 1 : R > 32 ? 32 : R;
        const int wide_in = nx % 16 == 0 && ((uintptr_t)occ & 15u) == 0;
        edt_pack<<<(unsigned)((rows + R - 1) / R), 256, (size_t)R * (p.words + 1) * 4, st>>>(
            occ, (uint2*)workspace, nx, ny, rows, p.words, R, wide_in);
        hipError_t e = hipGetLastError();
        p.n = ny;
        p.out = p.plane;
        if (e == hipSuccess)
            e = packed ? launch_tile<u16x2, kPlane, true>(p, ty, nz, st)
                       : launch_tile<uint32_t, kPlane, true>(p, ty, nz, st);
        p.n = nz;
        p.out = out;
        if (e == hipSuccess)
            e = packed ? launch_z<u16x2>(p, fout != nullptr, exact, tz, st)
                       : launch_z<uint32_t>(p, fout != nullptr, exact, tz, st);
        if (e != hipSuccess) return efail(-4, "sdfr_edt: launch failed: %s", hipGetErrorString(e));
        return 0;
    }
    // a line too long for LDS: the envelope walk
    int32_t* a = (int32_t*)workspace;
    int32_t* b = a + vox;
    uint64_t* v = (uint64_t*)((char*)workspace + edt_env_offset(nx, ny, nz));
    edt_rows<<<(int)((rows + 3) / 4), 256, 0, st>>>(occ, a, nx, rows);
    edt_cols<<<(int)((cols + 255) / 256), 256, 0, st>>>(a, b, v, nx, ny, nz);
    edt_slabs<<<(int)((lines + 255) / 256), 256, 0, st>>>(b, v, fout, hout, nx, ny, nz, cell2);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return efail(-4, "sdfr_edt: launch failed: %s", hipGetErrorString(e));
    return 0;
}

}  // extern "C"
