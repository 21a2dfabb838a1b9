// G^3 spatial grid over the Gaussians (getGridSamples, GaussianView.cpp:3870-4149;
// GetGsGrid / GetBoxesGsGrid + scans, cudakdtree.cu:403-451,508-553) and the
// density sample on its cells (the un-vendored forward3d_grid, called at
// GaussianView.cpp:4159-4186), for gfx950.
//
//   * scene AABB: device min/max reduction, then the float expansion rule on the host
//   * reorder: stable radix sort of the centre cells (the rank rule of
//     GaussianView.cpp:3904-3953 is exactly a stable sort by cell)
//   * lists: every Gaussian's (cell, id) pairs are emitted at a scanned offset, a
//     stable radix sort by cell yields per-cell lists in ascending id order —
//     the order of the reference's serial fill loop (GaussianView.cpp:4076-4100)
//   * density: one wave per valid cell, its falloffs times the Gaussians' SH rows
//     on the matrix cores
#pragma clang fp contract(off)
#include "common.hpp"
#include "grid.hpp"
#include "sort.hpp"

namespace arapgs {

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

__device__ __forceinline__ uint32_t ordered_bits(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t b) {
    return __uint_as_float((b & 0x80000000u) ? (b & 0x7fffffffu) : ~b);
}

// One atomic per workgroup and bound: 24,576 of them on one line (a workgroup of
// four waves each adding its own) took 0.28 ms whatever the points.
__global__ void __launch_bounds__(256) minmax_kernel(const float* __restrict__ pos, int64_t n,
                                                     uint32_t* __restrict__ mm) {
    __shared__ uint32_t s_lo[3], s_hi[3];
    if (threadIdx.x < 3) {
        s_lo[threadIdx.x] = 0xffffffffu;
        s_hi[threadIdx.x] = 0u;
    }
    __syncthreads();
    uint32_t lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const uint32_t b = ordered_bits(pos[3 * i + c]);
            lo[c] = min(lo[c], b);
            hi[c] = max(hi[c], b);
        }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[c] = min(lo[c], (uint32_t)__shfl_xor((int)lo[c], o));
            hi[c] = max(hi[c], (uint32_t)__shfl_xor((int)hi[c], o));
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMin(&s_lo[c], lo[c]);
            atomicMax(&s_hi[c], hi[c]);
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        atomicMin(&mm[threadIdx.x], s_lo[threadIdx.x]);
        atomicMax(&mm[3 + threadIdx.x], s_hi[threadIdx.x]);
    }
}

__global__ void minmax_init_kernel(uint32_t* __restrict__ mm) {
    if (threadIdx.x < 3) mm[threadIdx.x] = 0xffffffffu;
    else if (threadIdx.x < 6) mm[threadIdx.x] = 0u;
}

__global__ void decode_minmax_kernel(const uint32_t* __restrict__ mm, float* __restrict__ out) {
    if (threadIdx.x < 6) out[threadIdx.x] = from_ordered(mm[threadIdx.x]);
}

__device__ __forceinline__ int cell_coord(float p, float mn, float step) { return (int)floorf((p - mn) / step); }

__global__ void center_cell_kernel(const float* __restrict__ pos, int64_t n, GridGeom gg, uint64_t* __restrict__ keys,
                                   uint32_t* __restrict__ vals) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int x = cell_coord(pos[3 * i], gg.mn[0], gg.step);
    const int y = cell_coord(pos[3 * i + 1], gg.mn[1], gg.step);
    const int z = cell_coord(pos[3 * i + 2], gg.mn[2], gg.step);
    keys[i] = (uint64_t)(uint32_t)(x * gg.G * gg.G + y * gg.G + z);
    vals[i] = (uint32_t)i;
}

// alpha-cutoff AABB (GaussianView.cpp:3960-4019)
__global__ void aabb_kernel(const float* __restrict__ pos, const float* __restrict__ rot,
                            const float* __restrict__ scale, const float* __restrict__ opacity, int64_t n,
                            float* __restrict__ out) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    float q[4] = {rot[4 * g], rot[4 * g + 1], rot[4 * g + 2], rot[4 * g + 3]};
    quat_normalize(q);
    float R[3][3];
    quat_to_mat(q[0], q[1], q[2], q[3], R);
    const float cutoff = 1.0f / 255.0f;
    float s3[3] = {0.0f, 0.0f, 0.0f};
    if (opacity[g] > cutoff) {
        const float lg = (float)log((double)(cutoff / opacity[g]));
        const float f = __builtin_sqrtf(-2.0f * lg);
#pragma unroll
        for (int i = 0; i < 3; i++) s3[i] = f * (scale[3 * g + i] + 0.0f);
    }
    float lo[3], hi[3];
#pragma unroll
    for (int c = 0; c < 3; c++) lo[c] = hi[c] = pos[3 * g + c];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float off = R[c][d] * s3[d];
            const float a = pos[3 * g + c] + off, b = pos[3 * g + c] + (-off);
            lo[c] = fminf(lo[c], fminf(a, b));
            hi[c] = fmaxf(hi[c], fmaxf(a, b));
        }
#pragma unroll
    for (int c = 0; c < 3; c++) { out[6 * g + c] = lo[c]; out[6 * g + 3 + c] = hi[c]; }
}

__device__ __forceinline__ void box_range(const float* a, const GridGeom& gg, int lo[3], int hi[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
        lo[c] = max((int)(floorf((a[c] - gg.mn[c]) / gg.step) - (float)gg.padding), 0);
        hi[c] = min((int)(floorf((a[3 + c] - gg.mn[c]) / gg.step) + (float)gg.padding), gg.G - 1);
    }
}

__global__ void box_count_kernel(const float* __restrict__ aabbs, int64_t n, GridGeom gg, uint32_t* __restrict__ cnt) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    int lo[3], hi[3];
    box_range(aabbs + 6 * g, gg, lo, hi);
    const int nx = hi[0] - lo[0] + 1, ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
    cnt[g] = (nx > 0 && ny > 0 && nz > 0) ? (uint32_t)(nx * ny * nz) : 0u;
}

// 64-bit sum of the per-Gaussian cell counts (the total number of
// cell-Gaussian pairs, which may exceed 2^32 on large grids).
__global__ void sum_counts_kernel(const uint32_t* __restrict__ cnt, int64_t n, unsigned long long* __restrict__ out) {
    unsigned long long s = 0ull;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        s += cnt[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0 && s) atomicAdd(out, s);
}

// Pairs per x-slab of the grid (cells x*G^2 .. (x+1)*G^2-1): a Gaussian whose
// box spans ny*nz cells in y and z adds ny*nz to every slab its box crosses.
// Counted in LDS (s_slab: G counters) and added to memory once per workgroup
// and slab: with one memory atomic per Gaussian and slab, millions of them on G
// addresses, it took 22.4 ms at 1M Gaussians on a 64^3 grid, 0.03 ms this way.
__global__ void __launch_bounds__(256) slab_count_kernel(const float* __restrict__ aabbs, int64_t n, GridGeom gg,
                                                         unsigned long long* __restrict__ slab) {
    extern __shared__ unsigned long long s_slab[];
    for (int x = threadIdx.x; x < gg.G; x += blockDim.x) s_slab[x] = 0ull;
    __syncthreads();
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (int64_t)gridDim.x * blockDim.x) {
        int lo[3], hi[3];
        box_range(aabbs + 6 * g, gg, lo, hi);
        const int ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
        if (hi[0] < lo[0] || ny <= 0 || nz <= 0) continue;
        for (int x = lo[0]; x <= hi[0]; x++) atomicAdd(&s_slab[x], (unsigned long long)(ny * nz));
    }
    __syncthreads();
    for (int x = threadIdx.x; x < gg.G; x += blockDim.x)
        if (s_slab[x]) atomicAdd(&slab[x], s_slab[x]);
}

// Gaussians per cell as a prefix sum over the grid in x, y and z of the boxes'
// corner marks (+1 / -1 by parity; u32 arithmetic wraps, the sums do not): 8
// atomic adds per Gaussian instead of one per (cell, Gaussian) pair (0.56 ms at
// 1M Gaussians / 152M pairs).
__global__ void __launch_bounds__(256) box_corners_kernel(const float* __restrict__ aabbs, int64_t n, GridGeom gg,
                                                          uint32_t* __restrict__ cells) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    int lo[3], hi[3];
    box_range(aabbs + 6 * g, gg, lo, hi);
    if (hi[0] < lo[0] || hi[1] < lo[1] || hi[2] < lo[2]) return;
    const int64_t G = gg.G;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int x = c & 1 ? hi[0] + 1 : lo[0], y = c & 2 ? hi[1] + 1 : lo[1], z = c & 4 ? hi[2] + 1 : lo[2];
        if (x < G && y < G && z < G)
            atomicAdd(&cells[(x * G + y) * G + z], ((c ^ (c >> 1) ^ (c >> 2)) & 1) ? 0xffffffffu : 1u);
    }
}

// Inclusive prefix sums along z: one wave per row of G cells.
__global__ void __launch_bounds__(256) scan_rows_kernel(uint32_t* __restrict__ cells, int64_t rows, int G) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    uint32_t* r = cells + row * G;
    uint32_t carry = 0;
    for (int z0 = 0; z0 < G; z0 += 64) {
        const int z = z0 + lane;
        uint32_t v = z < G ? r[z] : 0u;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(v, o);
            if (lane >= o) v += t;
        }
        v += carry;
        if (z < G) r[z] = v;
        carry = __shfl(v, 63);
    }
}

// Inclusive prefix sums along an axis of stride `stride` (consecutive threads on
// consecutive z): lines are [outer][inner], inner < stride.
__global__ void __launch_bounds__(256) scan_lines_kernel(uint32_t* __restrict__ cells, int64_t lines, int64_t stride,
                                                         int G) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lines) return;
    uint32_t* p = cells + i / stride * stride * G + i % stride;
    uint32_t sum = 0;
    for (int k = 0; k < G; k++) {
        sum += p[k * stride];
        p[k * stride] = sum;
    }
}

// Cells of each Gaussian's box inside the slabs [x0, x1).
__global__ void box_count_slabs_kernel(const float* __restrict__ aabbs, int64_t n, GridGeom gg, int x0, int x1,
                                       uint32_t* __restrict__ cnt) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    int lo[3], hi[3];
    box_range(aabbs + 6 * g, gg, lo, hi);
    const int nx = min(hi[0], x1 - 1) - max(lo[0], x0) + 1;
    const int ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
    cnt[g] = (nx > 0 && ny > 0 && nz > 0) ? (uint32_t)(nx * ny * nz) : 0u;
}

// The pairs of the slabs [x0, x1): key = cell - x0*G^2 (32-bit), value = the
// Gaussian, written from offs[g] in ascending cell order. The 64 Gaussians of a
// wave own consecutive slots, which consecutive lanes write: the lane of slot j
// finds its Gaussian (the last of the 64 whose first slot is <= j) by a binary
// search over the lanes' first slots. A thread writing its own Gaussian's run
// (64 runs of ~600 bytes a wave) took 12.3 ms at 1M Gaussians / 152M pairs with
// an atomic count per pair, 0.41 ms this way.
// COUNT: every pair counts into its cell too (cell_counts_by_pair).
template <bool COUNT>
__global__ void __launch_bounds__(256) box_emit_slabs_kernel(const float* __restrict__ aabbs, int64_t n, GridGeom gg,
                                                             int x0, int x1, const uint32_t* __restrict__ offs,
                                                             uint32_t* __restrict__ keys,
                                                             uint32_t* __restrict__ vals,
                                                             uint32_t* __restrict__ cell_count) {
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool here = g < n;
    uint32_t first = 0xffffffffu, cnt = 0;
    int base = 0, ny = 1, nz = 1;  // first cell of the box, relative to the chunk
    if (here) {
        int lo[3], hi[3];
        box_range(aabbs + 6 * g, gg, lo, hi);
        const int xa = max(lo[0], x0), xb = min(hi[0], x1 - 1);
        first = offs[g];
        if (xb >= xa && hi[1] >= lo[1] && hi[2] >= lo[2]) {
            ny = hi[1] - lo[1] + 1;
            nz = hi[2] - lo[2] + 1;
            cnt = (uint32_t)((xb - xa + 1) * ny * nz);
            base = ((xa - x0) * gg.G + lo[1]) * gg.G + lo[2];
        }
    }
    const uint64_t hmask = __ballot(here);
    if (hmask == 0ull) return;
    const int last = 63 - __builtin_clzll(hmask);
    const uint32_t begin = __shfl(first, 0), end = __shfl(first + cnt, last);
    const uint32_t g0 = (uint32_t)((int64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63));
    // uniform trip count: every lane takes part in every shuffle
    for (uint32_t jb = begin; jb < end; jb += 64) {
        const uint32_t j = jb + (uint32_t)lane;
        int at = 0;
#pragma unroll
        for (int step = 32; step >= 1; step >>= 1) {
            const uint32_t f = __shfl(first, at + step);
            if (f <= j) at += step;
        }
        const uint32_t q = j - __shfl(first, at);
        const uint32_t w = (uint32_t)__shfl(nz, at), h = (uint32_t)__shfl(ny, at);
        const uint32_t b = (uint32_t)__shfl(base, at);
        if (j < end) {
            const uint32_t row = q / w, x = row / h;
            const uint32_t key = b + (x * (uint32_t)gg.G + (row - x * h)) * (uint32_t)gg.G + (q - row * w);
            keys[j] = key;
            vals[j] = g0 + (uint32_t)at;
            if (COUNT) atomicAdd(&cell_count[(uint32_t)(x0 * gg.G * gg.G) + key], 1u);
        }
    }
}

// 64-bit inclusive scan of the per-cell counts (tiles of 2048 cells): block
// sums, one-block scan of the sums, then each tile scanned with its offset.
constexpr int SCAN64_THREADS = 256;
constexpr int SCAN64_ITEMS = 8;
constexpr int SCAN64_TILE = SCAN64_THREADS * SCAN64_ITEMS;

__device__ __forceinline__ unsigned long long block_exclusive_scan64(unsigned long long v, unsigned long long* sh,
                                                                     unsigned long long* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long run = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
            const unsigned long long c = sh[w];
            sh[w] = run;
            run += c;
        }
        sh[16] = run;
    }
    __syncthreads();
    const unsigned long long r = sh[wave] + x - v;
    if (total) *total = sh[16];
    __syncthreads();
    return r;
}

__global__ void __launch_bounds__(SCAN64_THREADS) scan64_reduce_kernel(const uint32_t* __restrict__ in, int64_t n,
                                                                       unsigned long long* __restrict__ sums) {
    __shared__ unsigned long long sh[17];
    const int64_t base = (int64_t)blockIdx.x * SCAN64_TILE + (int64_t)threadIdx.x * SCAN64_ITEMS;
    unsigned long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN64_ITEMS; i++)
        if (base + i < n) s += in[base + i];
    unsigned long long tot;
    block_exclusive_scan64(s, sh, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN64_THREADS) scan64_blocks_kernel(unsigned long long* __restrict__ sums,
                                                                       int64_t nb) {
    __shared__ unsigned long long sh[17];
    unsigned long long carry = 0;
    for (int64_t base = 0; base < nb; base += SCAN64_THREADS) {
        const int64_t i = base + threadIdx.x;
        const unsigned long long v = i < nb ? sums[i] : 0ull;
        unsigned long long tot;
        const unsigned long long ex = block_exclusive_scan64(v, sh, &tot);
        if (i < nb) sums[i] = carry + ex;
        carry += tot;
    }
}

// prefix[c] = pairs in cells 0..c (inclusive), flags[c] = cell c holds any.
__global__ void __launch_bounds__(SCAN64_THREADS) scan64_apply_kernel(const uint32_t* __restrict__ in, int64_t n,
                                                                      const unsigned long long* __restrict__ block_off,
                                                                      int64_t* __restrict__ prefix,
                                                                      uint32_t* __restrict__ flags) {
    __shared__ unsigned long long sh[17];
    const int64_t base = (int64_t)blockIdx.x * SCAN64_TILE + (int64_t)threadIdx.x * SCAN64_ITEMS;
    uint32_t v[SCAN64_ITEMS];
    unsigned long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN64_ITEMS; i++) {
        v[i] = (base + i < n) ? in[base + i] : 0u;
        s += v[i];
    }
    unsigned long long run = block_exclusive_scan64(s, sh, nullptr) + block_off[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN64_ITEMS; i++) {
        run += v[i];
        if (base + i < n) {
            prefix[base + i] = (int64_t)run;
            flags[base + i] = v[i] ? 1u : 0u;
        }
    }
}

__global__ void compact_valid_kernel(const uint32_t* __restrict__ flags, const uint32_t* __restrict__ pos_ex,
                                     int64_t n, int* __restrict__ valid) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (flags[i]) valid[pos_ex[i]] = (int)i;
}

__global__ void samples_kernel(const int* __restrict__ valid, int64_t nv, GridGeom gg, float* __restrict__ samples) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nv * 64) return;
    const int64_t v = t / 64;
    const int s = (int)(t % 64);
    const int c = valid[v];
    const int G = gg.G;
    const int xi = c / (G * G), yi = (c - xi * G * G) / G, zi = c % G;
    const float interval = gg.step / 4;
    const float x0 = (float)((double)(gg.mn[0] + xi * gg.step) + 0.5 * (double)interval);
    const float y0 = (float)((double)(gg.mn[1] + yi * gg.step) + 0.5 * (double)interval);
    const float z0 = (float)((double)(gg.mn[2] + zi * gg.step) + 0.5 * (double)interval);
    const int sx = s / 16, sy = (s - sx * 16) / 4, sz = s % 4;
    samples[3 * t] = x0 + sx * interval;
    samples[3 * t + 1] = y0 + sy * interval;
    samples[3 * t + 2] = z0 + sz * interval;
}

// Density sample: a_g(x) = o_g exp(-1/2 d^T (Sigma_g + L)^-1 d), L = lpf I or
// the cell's adaptive filter, feature = sum a_g sh_g, opacity = sum a_g. The
// features of a cell are the product of its 64 x n falloffs and the n x 48 SH
// rows, so they run on the matrix cores: 4 sample tiles x 3 coefficient tiles, 32
// Gaussians a step, both operands split into three bf16 parts (split3; the six
// products above 2^-24, the same size of error as FP32 ones). One wave per cell.
// The lane that holds an operand computes it: lane l owns samples l % 16 + 16 t
// (positions in registers) and, of each step, Gaussians 8 (l / 16) .. + 7, so the
// falloffs never cross lanes, and the SH operands are read from memory in their
// operand layout (rows, 64 contiguous bytes of each per load).
// Bound by the vector instructions (88% of the SIMDs' issue), 14 and an
// exponential per falloff, 5.5 to split it and as many for an SH operand; bf16
// matrix instructions hide beside them but for 9 cycles each, where FP32 ones
// (v_mfma_f32_16x16x4f32, 32 cycles) do not overlap them at all. 500k Gaussians
// on a 64^3 grid (74M cell-Gaussian pairs): 11.1 ms with 48 vector FMAs a pair,
// 6.0 with FP32 matrix instructions, 5.3 so (two waves a SIMD: the same; four
// spill).
// BIG: the SH rows span 4 GiB or more (64-bit row addresses).
// L1: the cell's features and densities are compared with an aim instead of
// written: the signs of the differences and their weighted sum leave the kernel
// (64 + 192 bytes a sample against 192 + 4 written here and 388 read and 196
// written by a pass of its own, which took 3.1 ms at 89k cells).
constexpr int64_t DENSITY_BIG = (int64_t)0xffffffffu / 192;
template <bool BIG, bool L1>
__global__ void __launch_bounds__(64, 3) density_kernel(int64_t nv, const int* __restrict__ valid,
                                                     const int64_t* __restrict__ prefix, const int* __restrict__ list,
                                                     const float* __restrict__ samples, const float* __restrict__ pos,
                                                     const float* __restrict__ rot, const float* __restrict__ scale,
                                                     const float* __restrict__ opacity, const float* __restrict__ sh,
                                                     DensityFilter flt, float* __restrict__ feat,
                                                     float* __restrict__ opac, DensityAim aim) {
#pragma clang fp contract(fast)
    constexpr int B = 64;
    // mu (3), o | q00 2q01 2q02 q11 | 2q12 q22, scaled by -log2(e) / 2, SH row (byte
    // offset, or the Gaussian when BIG)
    __shared__ float4 s_p[B][3];
    const int64_t v = cell_of_block(blockIdx.x, nv);
    const int c = valid[v];
    const int64_t beg = c == 0 ? 0 : prefix[c - 1], end = prefix[c];
    const int lane = threadIdx.x, col = lane & 15, kq = lane >> 4;
    float x[4][3];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int k = 0; k < 3; k++) x[t][k] = samples[3 * (v * 64 + 16 * t + col) + k];
    float lf[6];
    density_filter_load(flt, v, lf);
    floatx4 acc[4][3];
    float aop[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        aop[t] = 0.0f;
#pragma unroll
        for (int u = 0; u < 3; u++) acc[t][u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // the parameters of up to B entries; those past the list's end get a falloff of zero times the last entry's row
    const auto stage = [&](int64_t b0, int m) {
        const int g = list[b0 + min(lane, m - 1)];
        float q[4] = {rot[4 * (int64_t)g], rot[4 * (int64_t)g + 1], rot[4 * (int64_t)g + 2], rot[4 * (int64_t)g + 3]};
        quat_normalize(q);
        float R[3][3];
        quat_to_mat(q[0], q[1], q[2], q[3], R);
        float s2[3], S[3][3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float sk = scale[3 * (int64_t)g + k];
            s2[k] = sk * sk;
        }
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++)
                S[i][j] = R[i][0] * s2[0] * R[j][0] + R[i][1] * s2[1] * R[j][1] + R[i][2] * s2[2] * R[j][2];
        density_filter_add(lf, S);
        const float c00 = S[1][1] * S[2][2] - S[1][2] * S[2][1];
        const float c01 = S[1][2] * S[2][0] - S[1][0] * S[2][2];
        const float c02 = S[1][0] * S[2][1] - S[1][1] * S[2][0];
        const float det = S[0][0] * c00 + S[0][1] * c01 + S[0][2] * c02;
        const float id = -0.72134752044448170f / det;
        const float id2 = 2.0f * id;
        s_p[lane][0] = make_float4(pos[3 * (int64_t)g], pos[3 * (int64_t)g + 1], pos[3 * (int64_t)g + 2],
                                   opacity[g]);
        s_p[lane][1] = make_float4(c00 * id, c01 * id2, c02 * id2, (S[0][0] * S[2][2] - S[0][2] * S[2][0]) * id);
        s_p[lane][2] = make_float4((S[0][2] * S[1][0] - S[0][0] * S[1][2]) * id2,
                                   (S[0][0] * S[1][1] - S[0][1] * S[1][0]) * id,
                                   __uint_as_float(BIG ? (uint32_t)g : 192u * (uint32_t)g), 0.0f);
        if (lane >= m) {
            s_p[lane][0] = s_p[lane][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            s_p[lane][2].x = s_p[lane][2].y = 0.0f;
        }
        __syncthreads();
    };
    for (int64_t b0 = beg; b0 < end; b0 += B) {
        const int m = (int)min((int64_t)B, end - b0);
        stage(b0, m);
        // 32 Gaussians a step; the SH operands of the second one are loaded before the first is computed
        const int steps = (m + 31) / 32;
        floatx8 d[3];
        const auto fetch = [&](int j) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t at = __float_as_uint(s_p[32 * j + 8 * kq + e][2].z);
                const char* r = reinterpret_cast<const char*>(sh) + (BIG ? 192 * (size_t)at : at);
#pragma unroll
                for (int u = 0; u < 3; u++) d[u][e] = reinterpret_cast<const float*>(r)[16 * u + col];
            }
        };
        fetch(0);
        for (int j = 0; j < steps; j++) {
            bf16x8 bs[3][3];
#pragma unroll
            for (int u = 0; u < 3; u++) split3(d[u], bs[u]);
            if (j + 1 < steps) fetch(j + 1);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                __builtin_amdgcn_sched_barrier(0);
                floatx8 a[2];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int k = 32 * j + 8 * kq + e;
                    const float4 p0 = s_p[k][0], p1 = s_p[k][1];
                    const float2 p2 = *reinterpret_cast<const float2*>(&s_p[k][2]);
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const float* xt = x[2 * h + t];
                        const float d0 = xt[0] - p0.x, d1 = xt[1] - p0.y, d2 = xt[2] - p0.z;
                        const float q = (p1.x * d0 + p1.y * d1 + p1.z * d2) * d0 + (p1.w * d1 + p2.x * d2) * d1 + p2.y * d2 * d2;
                        a[t][e] = p0.w * __builtin_amdgcn_exp2f(q);
                        aop[2 * h + t] += a[t][e];
                    }
                }
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
                    bf16x8 as[3];
                    split3(a[t], as);
#pragma unroll
                    for (int k = 0; k < 6; k++)
#pragma unroll
                        for (int u = 0; u < 3; u++)
                            acc[2 * h + t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as[pa[k]], bs[u][pb[k]],
                                                                                        acc[2 * h + t][u], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    // a sum that is not finite
    float odd = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int u = 0; u < 3; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) odd = __builtin_fmaf(acc[t][u][r], 0.0f, odd);
    if (__ballot(odd != 0.0f)) {  // (a NaN is not equal to zero)
        // The parts of an infinity, and of a value above bf16's largest, are no sum of it: the cell's sums as they
        // are, one Gaussian after the other.
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < 3; u++) acc[t][u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int64_t b0 = beg; b0 < end; b0 += B) {
            const int m = (int)min((int64_t)B, end - b0);
            stage(b0, m);
#pragma unroll 1
            for (int k = 0; k < m; k++) {
                const float4 p0 = s_p[k][0], p1 = s_p[k][1], p2 = s_p[k][2];
                const float* row = sh + 48 * (int64_t)list[b0 + k] + col;
                const float c[3] = {row[0], row[16], row[32]};
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float* xs = samples + 3 * (v * 64 + 16 * t + 4 * kq + r);
                        const float d0 = xs[0] - p0.x, d1 = xs[1] - p0.y, d2 = xs[2] - p0.z;
                        const float q = (p1.x * d0 + p1.y * d1 + p1.z * d2) * d0 + (p1.w * d1 + p2.x * d2) * d1 + p2.y * d2 * d2;
                        const float a = p0.w * __builtin_amdgcn_exp2f(q);
#pragma unroll
                        for (int u = 0; u < 3; u++) acc[t][u][r] = __builtin_fmaf(a, c[u], acc[t][u][r]);
                    }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        aop[t] += __shfl_xor(aop[t], 16);
        aop[t] += __shfl_xor(aop[t], 32);
    }
    // lane quarter t holds sample tile t
    const float dens = kq == 0 ? aop[0] : kq == 1 ? aop[1] : kq == 2 ? aop[2] : aop[3];
    // accumulator r of tile (t, u): sample 16 t + 4 (lane / 16) + r, coefficient 16 u + lane % 16
    if constexpr (L1) {
        static_assert(sizeof(s_p) >= 64 * 48, "the signs of 64 samples");
        int8_t* s_sign = reinterpret_cast<int8_t*>(s_p);
        const float* a = aim.feat + 48 * (v * 64 + 4 * kq) + col;
        double sum = 0.0;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int u = 0; u < 3; u++) {
                    const float d = acc[t][u][r] - a[48 * (16 * t + r) + 16 * u];
                    s_sign[48 * (16 * t + 4 * kq + r) + 16 * u + col] = d > 0.0f ? 1 : d < 0.0f ? -1 : 0;
                    sum += fabs((double)d);
                }
        const float d = dens - aim.dens[v * 64 + lane];
        sum += (double)aim.w * fabs((double)d);
        __syncthreads();
        const int4* row = reinterpret_cast<const int4*>(s_sign + 48 * lane);
        int4* out = reinterpret_cast<int4*>(aim.signs + DENSITY_SIGNS * (v * 64 + lane));
        out[0] = row[0];
        out[1] = row[1];
        out[2] = row[2];
        out[3] = make_int4(d > 0.0f ? 1 : d < 0.0f ? 0xff : 0, 0, 0, 0);
#pragma unroll
        for (int k = 32; k > 0; k >>= 1) sum += __shfl_xor(sum, k);
        if (lane == 0) {
            aim.cell_sum[v] = sum;
            aim.cell_loss[v] = (float)sum;
        }
        return;
    }
    float* o = feat + 48 * (v * 64 + 4 * kq) + col;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int u = 0; u < 3; u++) o[48 * (16 * t + r) + 16 * u] = acc[t][u][r];
    opac[v * 64 + lane] = dens;
}

// The sum of the cells' losses, added to *loss.
__global__ void __launch_bounds__(256) cell_sum_kernel(const double* __restrict__ cell_sum, int64_t nv,
                                                       double* __restrict__ loss) {
    __shared__ double s_red[4];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += (int64_t)gridDim.x * blockDim.x)
        acc += cell_sum[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) unsafeAtomicAdd(loss, s_red[0] + s_red[1] + s_red[2] + s_red[3]);
}

// GetAdaLpfRatio (GaussianView.cpp:4670-4749), one thread per valid cell. The
// cell's samples are a 4x4x4 block (sample x*16 + y*4 + z); corner c has
// offsets q_c = (c&1, (c>>1)&1, (c>>2)&1) and the sample at 48 q_x + 12 q_y +
// 3 q_z. With p_c = (x_c - x_0) / 3, the reference solves the 24 x 9 least
// squares min sum_c |M q_c - p_c|^2 by the normal equations; they decouple
// per row of M, with Q Q^T = 2 I + 2 11^T over the cube's corners, whose
// inverse is 3/8 on the diagonal and -1/8 off it, so M = (P Q^T)(Q Q^T)^-1
// in closed form (evaluated in double). out = lpf_param * M M^T.
__global__ void __launch_bounds__(256) ada_lpf_kernel(int64_t nv, const float* __restrict__ samples,
                                                      float lpf_param, float* __restrict__ out) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const float* x = samples + 3 * 64 * v;
    double PQ[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};  // P Q^T
    for (int c = 1; c < 8; c++) {
        const int qx = c & 1, qy = (c >> 1) & 1, qz = (c >> 2) & 1;
        const float* xc = x + 3 * (48 * qx + 12 * qy + 3 * qz);
        for (int j = 0; j < 3; j++) {
            const double pj = (double)((xc[j] - x[j]) / 3.0f);
            if (qx) PQ[j][0] += pj;
            if (qy) PQ[j][1] += pj;
            if (qz) PQ[j][2] += pj;
        }
    }
    double M[3][3];
    for (int j = 0; j < 3; j++) {
        const double sum = PQ[j][0] + PQ[j][1] + PQ[j][2];
        for (int k = 0; k < 3; k++) M[j][k] = 0.5 * PQ[j][k] - 0.125 * sum;
    }
    double L[3][3];
    for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) L[i][j] = (double)lpf_param * (M[i][0] * M[j][0] + M[i][1] * M[j][1] + M[i][2] * M[j][2]);
    float* o = out + 6 * v;
    o[0] = (float)L[0][0]; o[1] = (float)L[1][1]; o[2] = (float)L[2][2];
    o[3] = (float)L[0][1]; o[4] = (float)L[0][2]; o[5] = (float)L[1][2];
}

__global__ void zero_words_kernel(uint32_t* __restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

}  // namespace

int launch_minmax(const float* pos, int64_t n, uint32_t* mm_ws, float* out6, hipStream_t st) {
    hipLaunchKernelGGL(minmax_init_kernel, dim3(1), dim3(64), 0, st, mm_ws);
    hipLaunchKernelGGL(minmax_kernel, dim3(std::min<unsigned>(nblk(n, 256), 512)), dim3(256), 0, st, pos, n, mm_ws);
    hipLaunchKernelGGL(decode_minmax_kernel, dim3(1), dim3(64), 0, st, mm_ws, out6);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_center_cells(const float* pos, int64_t n, const GridGeom& gg, uint64_t* keys, uint32_t* vals,
                        hipStream_t st) {
    hipLaunchKernelGGL(center_cell_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, pos, n, gg, keys, vals);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_aabbs(const float* pos, const float* rot, const float* scale, const float* opacity, int64_t n, float* out,
                 hipStream_t st) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(aabb_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, pos, rot, scale, opacity, n, out);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_box_count(const float* aabbs, int64_t n, const GridGeom& gg, uint32_t* cnt, hipStream_t st) {
    hipLaunchKernelGGL(box_count_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, aabbs, n, gg, cnt);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_sum_counts(const uint32_t* cnt, int64_t n, unsigned long long* out, hipStream_t st) {
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, st, reinterpret_cast<uint32_t*>(out), (int64_t)2);
    if (n > 0)
        hipLaunchKernelGGL(sum_counts_kernel, dim3(std::min<unsigned>(nblk(n, 256), 1024u)), dim3(256), 0, st, cnt, n,
                           out);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_slab_counts(const float* aabbs, int64_t n, const GridGeom& gg, unsigned long long* slab, hipStream_t st) {
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(256), 0, st, reinterpret_cast<uint32_t*>(slab),
                       (int64_t)2 * gg.G);
    if (n > 0)
        hipLaunchKernelGGL(slab_count_kernel, dim3(std::min<unsigned>(nblk(n, 256), 1024u)), dim3(256),
                           sizeof(unsigned long long) * (size_t)gg.G, st, aabbs, n, gg, slab);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_cell_counts(const float* aabbs, int64_t n, const GridGeom& gg, uint64_t npairs, uint32_t* cell_count,
                       hipStream_t st) {
    const int64_t G = gg.G, G2 = G * G;
    hipLaunchKernelGGL(zero_words_kernel, dim3(std::min<unsigned>(nblk(G2 * G, 256), 4096)), dim3(256), 0, st,
                       cell_count, G2 * G);
    if (n > 0 && !cell_counts_by_pair(gg, npairs)) {
        hipLaunchKernelGGL(box_corners_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, aabbs, n, gg, cell_count);
        hipLaunchKernelGGL(scan_rows_kernel, dim3(nblk(G2, 4)), dim3(256), 0, st, cell_count, G2, gg.G);
        hipLaunchKernelGGL(scan_lines_kernel, dim3(nblk(G2, 256)), dim3(256), 0, st, cell_count, G2, G, gg.G);
        hipLaunchKernelGGL(scan_lines_kernel, dim3(nblk(G2, 256)), dim3(256), 0, st, cell_count, G2, G2, gg.G);
    }
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_box_count_slabs(const float* aabbs, int64_t n, const GridGeom& gg, int x0, int x1, uint32_t* cnt,
                           hipStream_t st) {
    hipLaunchKernelGGL(box_count_slabs_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, aabbs, n, gg, x0, x1, cnt);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_box_emit_slabs(const float* aabbs, int64_t n, const GridGeom& gg, uint64_t npairs, int x0, int x1,
                          const uint32_t* offs, uint32_t* keys, uint32_t* vals, uint32_t* cell_count, hipStream_t st) {
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nblk(n, 256)), dim3(256), 0, st, aabbs, n, gg, x0, x1, offs, keys, vals,
                           cell_count);
    };
    if (cell_counts_by_pair(gg, npairs)) launch(box_emit_slabs_kernel<true>);
    else launch(box_emit_slabs_kernel<false>);
    HIP_RET(hipGetLastError());
    return 0;
}

size_t cell_prefix_workspace_words(int64_t gc) { return 2 * (size_t)((gc + SCAN64_TILE - 1) / SCAN64_TILE) + 2; }

int launch_cell_prefix(const uint32_t* cell_count, int64_t gc, int64_t* prefix, uint32_t* flags, uint32_t* ws,
                       hipStream_t st) {
    const int64_t nb = (gc + SCAN64_TILE - 1) / SCAN64_TILE;
    if (nb == 0) return 0;
    unsigned long long* sums = reinterpret_cast<unsigned long long*>(ws);
    hipLaunchKernelGGL(scan64_reduce_kernel, dim3((unsigned)nb), dim3(SCAN64_THREADS), 0, st, cell_count, gc, sums);
    hipLaunchKernelGGL(scan64_blocks_kernel, dim3(1), dim3(SCAN64_THREADS), 0, st, sums, nb);
    hipLaunchKernelGGL(scan64_apply_kernel, dim3((unsigned)nb), dim3(SCAN64_THREADS), 0, st, cell_count, gc,
                       (const unsigned long long*)sums, prefix, flags);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_compact_valid(const uint32_t* flags, const uint32_t* pos_ex, int64_t gc, int* valid, hipStream_t st) {
    hipLaunchKernelGGL(compact_valid_kernel, dim3(nblk(gc, 256)), dim3(256), 0, st, flags, pos_ex, gc, valid);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_samples(const int* valid, int64_t nv, const GridGeom& gg, float* samples, hipStream_t st) {
    if (nv == 0) return 0;
    hipLaunchKernelGGL(samples_kernel, dim3(nblk(nv * 64, 256)), dim3(256), 0, st, valid, nv, gg, samples);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_density(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                   const float* samples, const float* pos, const float* rot, const float* scale, const float* opacity, const float* sh,
                   DensityFilter flt, float* feat, float* opac, hipStream_t st) {
    if (nv == 0) return 0;
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nv), dim3(64), 0, st, nv, valid, prefix, list, samples, pos, rot, scale,
                           opacity, sh, flt, feat, opac, DensityAim{});
    };
    if (n_gauss > DENSITY_BIG) launch(density_kernel<true, false>);
    else launch(density_kernel<false, false>);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_density_l1(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                      const float* samples, const float* pos, const float* rot, const float* scale,
                      const float* opacity, const float* sh, DensityFilter flt, const DensityAim& aim, double* loss,
                      hipStream_t st) {
    if (nv == 0) return 0;
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nv), dim3(64), 0, st, nv, valid, prefix, list, samples, pos, rot, scale,
                           opacity, sh, flt, (float*)nullptr, (float*)nullptr, aim);
    };
    if (n_gauss > DENSITY_BIG) launch(density_kernel<true, true>);
    else launch(density_kernel<false, true>);
    if (loss)
        hipLaunchKernelGGL(cell_sum_kernel, dim3(std::min<unsigned>(nblk(nv, 1024), 64)), dim3(256), 0, st,
                           aim.cell_sum, nv, loss);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_ada_lpf(int64_t nv, const float* samples, float lpf_param, float* out, hipStream_t st) {
    if (nv == 0) return 0;
    hipLaunchKernelGGL(ada_lpf_kernel, dim3(nblk(nv, 256)), dim3(256), 0, st, nv, samples, lpf_param, out);
    HIP_RET(hipGetLastError());
    return 0;
}

}  // namespace arapgs
