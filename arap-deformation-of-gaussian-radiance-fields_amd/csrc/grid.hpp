// Grid / density launchers (grid.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace arapgs {

struct GridGeom {
    float mn[3];
    float step;
    int G;
    int padding;
};

// The low-pass filter added to a density Gaussian's covariance: lpf I, or,
// when ada is set, the valid cell's own symmetric matrix ada[6v .. 6v+5]
// (xx, yy, zz, xy, xz, yz; the adaptive filter of GetAdaLpfRatio,
// GaussianView.cpp:4670-4749). With ada set, the density backward hands
// dL/dSigma (not dL/dSigma^-1) to the per-Gaussian kernels.
struct DensityFilter {
    float lpf;
    const float* ada;
};

typedef float floatx4 __attribute__((ext_vector_type(4)));  // a 16x16 matrix-core accumulator

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx8 __attribute__((ext_vector_type(8)));

// x = p[0] + p[1] + p[2] to 24 bits: each part the bf16 nearest to what is left.
// The parts are widened out of their packed pairs (a shift or a mask each):
// converted element by element, the compiler rounds every one a second time.
__device__ __forceinline__ void split3(floatx8 x, bf16x8 (&p)[3]) {
    typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int k = 0; k < 3; k++) {
        p[k] = __builtin_convertvector(x, bf16x8);
        if (k == 2) break;
        const uintx4 u = __builtin_bit_cast(uintx4, p[k]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            x[2 * i] -= __uint_as_float(u[i] << 16);
            x[2 * i + 1] -= __uint_as_float(u[i] & 0xffff0000u);
        }
    }
}

// The valid cell of a workgroup of the density kernels. Workgroups go to the 8
// XCDs in turn, and neighbouring cells list mostly the same Gaussians, so runs
// of CELL_RUN consecutive cells are given to one XCD (its L2 then reads a
// Gaussian's row once for the run instead of every XCD reading it); short runs
// keep the XCDs' loads even where dense and thin regions alternate (density of
// 500k Gaussians with FP32 matrix instructions: runs of 32, 128, 512, 2048 cells
// 5.89, 6.01, 6.82, 6.00 ms).
// A permutation of [0, nv).
constexpr int CELL_RUN = 32;
__device__ __forceinline__ int64_t cell_of_block(int64_t b, int64_t nv) {
    if (b >= nv / (8 * CELL_RUN) * (8 * CELL_RUN)) return b;
    const int64_t q = b / 8;
    return (q / CELL_RUN * 8 + b % 8) * CELL_RUN + q % CELL_RUN;
}

// The filter of valid cell v as (xx, yy, zz, xy, xz, yz), and its sum with a
// covariance S.
__device__ __forceinline__ void density_filter_load(const DensityFilter& f, int64_t v, float L[6]) {
#pragma unroll
    for (int k = 0; k < 6; k++) L[k] = f.ada ? f.ada[6 * v + k] : (k < 3 ? f.lpf : 0.0f);
}
__device__ __forceinline__ void density_filter_add(const float L[6], float S[3][3]) {
    S[0][0] += L[0]; S[1][1] += L[1]; S[2][2] += L[2];
    S[0][1] += L[3]; S[1][0] += L[3];
    S[0][2] += L[4]; S[2][0] += L[4];
    S[1][2] += L[5]; S[2][1] += L[5];
}

int launch_minmax(const float* pos, int64_t n, uint32_t* mm_ws, float* out6, hipStream_t st);
int launch_center_cells(const float* pos, int64_t n, const GridGeom& gg, uint64_t* keys, uint32_t* vals,
                        hipStream_t st);
int launch_aabbs(const float* pos, const float* rot, const float* scale, const float* opacity, int64_t n, float* out,
                 hipStream_t st);
int launch_box_count(const float* aabbs, int64_t n, const GridGeom& gg, uint32_t* cnt, hipStream_t st);
// *out (device, 8 bytes) = the 64-bit sum of cnt[0..n).
int launch_sum_counts(const uint32_t* cnt, int64_t n, unsigned long long* out, hipStream_t st);
// Pairs per emit + sort pass of the cell-list build (temporary buffers of
// 16 bytes per pair), and the most one x-slab may hold (32-bit offsets).
constexpr unsigned long long GRID_CHUNK_PAIRS = 1ull << 28;
constexpr unsigned long long GRID_CHUNK_PAIRS_MAX = 0x7fffffffull;

// Cell lists are built in chunks of whole x-slabs (cells x*G^2 .. (x+1)*G^2-1)
// so that each chunk's pairs fit 32-bit sort offsets; the per-cell prefix is
// 64-bit. slab: 2*G words (G u64 pair counts).
int launch_slab_counts(const float* aabbs, int64_t n, const GridGeom& gg, unsigned long long* slab, hipStream_t st);
// Whether a grid's pairs (npairs in all) are counted one by one as they are
// emitted; more of them, or more on a cell (their atomic adds take turns), are
// counted from the boxes' corners, whose scans take four launches. A build from
// the corners and pair by pair: 1.5k pairs on 64^3 326 and 255 us, 3.7M 750 and
// 657 us, 213k pairs on 4^3 310 and 458 us, 47M on 8^3 3.1 and 10 ms.
inline bool cell_counts_by_pair(const GridGeom& gg, uint64_t npairs) {
    return npairs <= std::min<uint64_t>(1ull << 22, 1024ull * gg.G * gg.G * gg.G);
}
// cell_count[c] (u32[G^3]) = Gaussians whose boxes cover cell c; only cleared
// where the emission counts (cell_counts_by_pair).
int launch_cell_counts(const float* aabbs, int64_t n, const GridGeom& gg, uint64_t npairs, uint32_t* cell_count,
                       hipStream_t st);
int launch_box_count_slabs(const float* aabbs, int64_t n, const GridGeom& gg, int x0, int x1, uint32_t* cnt,
                           hipStream_t st);
int launch_box_emit_slabs(const float* aabbs, int64_t n, const GridGeom& gg, uint64_t npairs, int x0, int x1,
                          const uint32_t* offs, uint32_t* keys, uint32_t* vals, uint32_t* cell_count, hipStream_t st);
// prefix[c] (int64) = pairs in cells 0..c, flags[c] = 1 if cell c holds any;
// ws holds cell_prefix_workspace_words(gc) words.
size_t cell_prefix_workspace_words(int64_t gc);
int launch_cell_prefix(const uint32_t* cell_count, int64_t gc, int64_t* prefix, uint32_t* flags, uint32_t* ws,
                       hipStream_t st);
int launch_compact_valid(const uint32_t* flags, const uint32_t* pos_ex, int64_t gc, int* valid, hipStream_t st);
int launch_samples(const int* valid, int64_t nv, const GridGeom& gg, float* samples, hipStream_t st);
// n_gauss: the Gaussians the grid's lists may name.
int launch_density(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                   const float* samples, const float* pos, const float* rot, const float* scale, const float* opacity, const float* sh,
                   DensityFilter flt, float* feat, float* opac, hipStream_t st);

// What a density sample is compared with: features (nv x 64 x 48) and densities
// (nv x 64), the densities' weight, and where the result goes: per sample a row
// of DENSITY_SIGNS bytes (the 48 signs of the differences and the density's; the
// rest 0; 16-byte aligned) and per cell sum |feature difference| + w sum
// |density difference|.
constexpr int DENSITY_SIGNS = 64;
struct DensityAim {
    const float* feat;
    const float* dens;
    float w;
    int8_t* signs;
    double* cell_sum;
    float* cell_loss;
};
// The density sample compared with an aim; *loss (may be null) += the sum over
// the cells.
int launch_density_l1(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                      const float* samples, const float* pos, const float* rot, const float* scale,
                      const float* opacity, const float* sh, DensityFilter flt, const DensityAim& aim, double* loss,
                      hipStream_t st);
// GetAdaLpfRatio (GaussianView.cpp:4670-4749) for nv valid cells: the linear
// map M that best carries the unit cube's corners to the cell's 8 corner
// samples (relative to sample 0, over the 3 sample intervals), and
// out[6v ..] = lpf_param * M M^T.
int launch_ada_lpf(int64_t nv, const float* samples, float lpf_param, float* out, hipStream_t st);

}  // namespace arapgs
