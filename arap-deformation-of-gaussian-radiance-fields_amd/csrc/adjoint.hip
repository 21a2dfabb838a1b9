// Reverse mode of the deform -> density-sample -> render chain (gfx950).
//
// Forward chain, per Gaussian (rest mean mu0, rest rotation q0, rest scale
// s0, SH c0): six end points e = mu0 +- R(q0/|q0|)[:,i] (s0_i + pad) coeff
// (GetEndPoints, GaussianView.cpp:4643-4668), each blended by its K nodes
// e' = sum_j w_j (R_j (e - g_j) + t_j + g_j) (predict_mesh, Deform.hpp:230-247),
// then the six-point update (UpdateAsSixPointsWithdrawBad,
// GaussianView.cpp:3081-3166): mu' = mean of e', R, S = polar of
// M = [(e'_{i+} - e'_{i-}) / 2], q' = quat(R) / |quat(R)|,
// s'_i = S_ii / ((s0_i + pad) coeff) s0_i, c' = SH rotation of c0 by
// R(normalise(q' q0^-1)). Samples x are blended the same way. The renderer
// and the density sampler read (mu', q', s', c') and the blended samples.
//
// The kernels here take the output-side gradients (from the renderer's
// backward and the density backward below) back to the node transforms
// (R_j, t_j), q0 and s0:
//   density_rows_kernel       the density's parameters of every Gaussian as
//                             48-byte rows
//   density_backward_kernel   one workgroup per valid cell (density_plain_backward_kernel:
//                             one wave, for operands that are not split): sample gradients
//                             (owned by the cell) and per-(cell, Gaussian)
//                             atomic adds of d mu', d Q (inverse covariance)
//                             and d c'
//   six_point_backward_kernel one thread per Gaussian: density covariance
//                             gradient to (q', s'), SH rotation, quaternion,
//                             polar and centre adjoints, blend adjoint to the
//                             rest end points and the end-point adjoint to
//                             (q0, s0); writes d e' per end point
//   node_gather_kernel        one workgroup per node over the node's entries
//                             of the (end point | sample) x slot inverse
//                             index: d R_j, d t_j in FP64, no atomics
#pragma clang fp contract(off)
#include "adjoint.hpp"
#include "common.hpp"
#include "sort.hpp"

namespace arapgs {

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

__global__ void zero_f32_kernel(float* __restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

__global__ void set_word_kernel(int* __restrict__ p) {
    if (threadIdx.x == 0) *p = 1;
}

// Covariance of a density Gaussian, Sigma = R(q/|q|) diag(s^2) R^T, packed (00,
// 11, 22, 01, 02, 12).
__device__ __forceinline__ void density_cov(const float* __restrict__ rot, const float* __restrict__ scale, int64_t g,
                                            float S[6]) {
#pragma clang fp contract(fast)
    float q[4] = {rot[4 * g], rot[4 * g + 1], rot[4 * g + 2], rot[4 * g + 3]};
    quat_normalize(q);
    float R[3][3];
    quat_to_mat(q[0], q[1], q[2], q[3], R);
    const int ii[6] = {0, 1, 2, 0, 0, 1}, jj[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int c = 0; c < 6; c++) {
        float a = 0.0f;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float sk = scale[3 * g + k];
            a += R[ii[c]][k] * sk * sk * R[jj[c]][k];
        }
        S[c] = a;
    }
}

// Q = (Sigma + L)^-1 by cofactors, both packed as above (L: density_filter_load's).
__device__ __forceinline__ void density_inverse(const float S[6], const float L[6], float Q[6]) {
#pragma clang fp contract(fast)
    const float a = S[0] + L[0], b = S[1] + L[1], c = S[2] + L[2], d = S[3] + L[3], e = S[4] + L[4], f = S[5] + L[5];
    const float c00 = b * c - f * f, c01 = f * e - d * c, c02 = d * f - b * e;
    const float id = 1.0f / (a * c00 + d * c01 + e * c02);
    Q[0] = c00 * id;
    Q[1] = (a * c - e * e) * id;
    Q[2] = (a * b - d * d) * id;
    Q[3] = c01 * id;
    Q[4] = c02 * id;
    Q[5] = (e * d - a * f) * id;
}

// dSigma = -Q dQ Q for Q = Sigma^-1, both symmetric and packed (00, 11, 22,
// 01, 02, 12); the off-diagonal entries of dq6 and of the result count both
// symmetric entries (dL/dX01 + dL/dX10).
__device__ __forceinline__ void dinv_to_dsigma(const float Qv[6], const float dq6[6], float ds6[6]) {
    const float Qm[3][3] = {{Qv[0], Qv[3], Qv[4]}, {Qv[3], Qv[1], Qv[5]}, {Qv[4], Qv[5], Qv[2]}};
    const float dQ[3][3] = {{dq6[0], 0.5f * dq6[3], 0.5f * dq6[4]},
                            {0.5f * dq6[3], dq6[1], 0.5f * dq6[5]},
                            {0.5f * dq6[4], 0.5f * dq6[5], dq6[2]}};
    float tmp[3][3], dS[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) tmp[i][j] = dQ[i][0] * Qm[0][j] + dQ[i][1] * Qm[1][j] + dQ[i][2] * Qm[2][j];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) dS[i][j] = -(Qm[i][0] * tmp[0][j] + Qm[i][1] * tmp[1][j] + Qm[i][2] * tmp[2][j]);
    ds6[0] = dS[0][0]; ds6[1] = dS[1][1]; ds6[2] = dS[2][2];
    ds6[3] = dS[0][1] + dS[1][0]; ds6[4] = dS[0][2] + dS[2][0]; ds6[5] = dS[1][2] + dS[2][1];
}

// Operands from here on are not split into bf16 parts (density_backward_kernel):
// the parts of an infinity, and of a value above bf16's largest, are no sum of it,
// and large products of parts overflow one by one.
constexpr float SPLIT_MOST = 0x1p60f;
__device__ __forceinline__ bool split_large(const float4& x) {
    return fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))) >= SPLIT_MOST;
}

// The density's per-Gaussian parameters as rows of three float4: mu (3), o |
// (00, 11, 22, 01) (02, 12, -, -) of Q = (Sigma + lpf I)^-1, or of Sigma itself
// where the filter is the cell's own. *large = 1 where an SH coefficient or an
// opacity is from SPLIT_MOST on.
__global__ void __launch_bounds__(256) density_rows_kernel(int64_t N, const float* __restrict__ pos,
                                                           const float* __restrict__ rot,
                                                           const float* __restrict__ scale,
                                                           const float* __restrict__ opacity,
                                                           const float* __restrict__ sh, DensityFilter flt,
                                                           float4* __restrict__ rows, int* __restrict__ large) {
    const int64_t g0 = (int64_t)blockIdx.x * 256, g = g0 + threadIdx.x;
    const float4* c4 = reinterpret_cast<const float4*>(sh + 48 * g0);
    const int n4 = 12 * (int)min<int64_t>(256, N - g0);
    bool big = false;
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const int i = 256 * k + threadIdx.x;
        if (i < n4) big = big || split_large(c4[i]);
    }
    if (big || (g < N && fabsf(opacity[g]) >= SPLIT_MOST)) *large = 1;
    if (g >= N) return;
    float S[6];
    density_cov(rot, scale, g, S);
    if (!flt.ada) {
        float L[6], Q[6];
        density_filter_load(flt, 0, L);
        density_inverse(S, L, Q);
#pragma unroll
        for (int k = 0; k < 6; k++) S[k] = Q[k];
    }
    rows[3 * g] = make_float4(pos[3 * g], pos[3 * g + 1], pos[3 * g + 2], opacity[g]);
    rows[3 * g + 1] = make_float4(S[0], S[1], S[2], S[3]);
    rows[3 * g + 2] = make_float4(S[4], S[5], 0.0f, 0.0f);
}

// c[i] += a[i] b[i] for operands split in three: the six products above 2^-24 of
// the largest, smallest first (the same size of error as FP32 products); the N
// independent accumulators in turn hide each other's latency.
template <int N>
__device__ __forceinline__ void mfma_split3(const bf16x8 (&a)[N][3], const bf16x8 (&b)[N][3], floatx4 (&c)[N]) {
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int k = 0; k < 6; k++)
#pragma unroll
        for (int i = 0; i < N; i++)
            c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa[k]], b[i][pb[k]], c[i], 0, 0, 0);
}

// Adds a wave's 16 Gaussians (lane l: g of Gaussian l % 16, of which m are
// there) to their rows: acc[u][r], coefficient 16 u + col of Gaussian 4 quad + r
// (features: not all zero), and the ten values out, the same in the four lanes of
// a Gaussian. s_par: the wave's scratch.
__device__ __forceinline__ void density_row_add(float* __restrict__ gacc, int g, int m, bool features,
                                                const floatx4 (&acc)[3], const float (&out)[10],
                                                float (*s_par)[17]) {
    const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
    // one Gaussian's ten values in the lanes of one quarter, as the accumulators hold its coefficients
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float w0 = out[4 * k], w1 = out[min(4 * k + 1, 9)], w2 = out[min(4 * k + 2, 9)], w3 = out[min(4 * k + 3, 9)];
        const float w01 = quad & 1 ? w1 : w0, w23 = quad & 1 ? w3 : w2;
        s_par[col][4 * k + quad] = quad & 2 ? w23 : w01;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float par[4];
#pragma unroll
    for (int r = 0; r < 4; r++) par[r] = s_par[4 * quad + r][col];
    // Swapping the odd quarters of one register with the even ones of another
    // leaves 32 neighbouring values of Gaussian 4 (quad & 2) + r in the first,
    // of the one four further on in the second.
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j0 = 4 * (quad & 2) + r, j1 = j0 + 4;
        float* d0 = gacc + 64 * (int64_t)__shfl(g, j0) + 16 * (quad & 1) + col;
        float* d1 = gacc + 64 * (int64_t)__shfl(g, j1) + 16 * (quad & 1) + col;
        const bool has0 = j0 < m, has1 = j1 < m;
        if (features) {
            const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[0][r]), __float_as_uint(acc[1][r]), false,
                                                            false);
            if (has0) unsafeAtomicAdd(d0, __uint_as_float(w[0]));
            if (has1) unsafeAtomicAdd(d1, __uint_as_float(w[1]));
        }
        const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[2][r]), __float_as_uint(par[r]), false, false);
        const bool used = (quad & 1) == 0 || col < 10;
        if (has0 && used) unsafeAtomicAdd(d0 + 32, __uint_as_float(w[0]));
        if (has1 && used) unsafeAtomicAdd(d1 + 32, __uint_as_float(w[1]));
    }
}

// a_gs = o_g exp(-q/2), q = d^T Q d, d = x_s - mu_g; feat_s = sum_g a_gs c_g,
// dens_s = sum_g a_gs. With da = dL/dfeat_s . c_g + dL/ddens_s:
//   dL/dc_g += a dL/dfeat_s,  dL/dq = -a da / 2,  dL/dQ += dL/dq d d^T,
//   dL/dx_s += 2 dL/dq Q d,   dL/dmu_g -= 2 dL/dq Q d.
// da (64 x 16 Gaussians, over 48 coefficients + the density) and dL/dc (16 x 48,
// over 64 samples) are matrix products and run on the matrix cores. FP32 matrix
// instructions hold up the vector ones (the falloffs and the sums over d), bf16
// ones hardly do, so the operands are split into three bf16 parts
// (mfma_split3). One workgroup of four waves per cell: dL/dfeat is split once
// into both products' operand layouts in LDS (43 KB: three workgroups per CU),
// then each wave takes 16 Gaussians at a time. Lane l owns Gaussian l % 16 and
// samples 16 t + 4 (l / 16) + r: the layout in which the first product's
// accumulators hold da is, with the sample index permuted alike on both sides,
// the one in which the second takes its falloffs, so nothing crosses lanes but
// the sums over the four lanes of a Gaussian.
// gacc, N rows of 64: d c (48), d mu (3), d Q (q00, q11, q22, then q01, q02, q12
// each counted for both symmetric entries; with an adaptive filter, whose Q
// differs per cell, d Sigma = -Q dQ Q in the same packing instead), d o; the
// last 6 are not used. The atomic adds are paid by the request of up to 64
// contiguous bytes, at most 20 G/s wherever the rows lie and whichever XCD asks: with 3
// of 64 bytes and 3 of 16 a pair they bounded the kernel, so the lanes are
// arranged for 4 of 64 in rows of two cache lines (1M Gaussians on 64^3, 223M
// pairs: 43.9 -> 29.8 ms, 16.8 without any atomics; 300k with sample gradients
// 14.5 -> 10.4 ms, 8.6 without).
template <bool ADA, bool SAMP>
__global__ void __launch_bounds__(256, SAMP ? 2 : 3) density_backward_kernel(int64_t nv, const int* __restrict__ valid,
                                                                  const int64_t* __restrict__ prefix,
                                                                  const int* __restrict__ list,
                                                                  const float* __restrict__ samples,
                                                                  const float4* __restrict__ rows,
                                                                  const float* __restrict__ sh, DensityFilter flt,
                                                                  const float* __restrict__ dfeat,
                                                                  const float* __restrict__ ddens,
                                                                  float* __restrict__ gsamp, float* __restrict__ gacc,
                                                                  const int* __restrict__ large,
                                                                  uint8_t* __restrict__ cell_large) {
#pragma clang fp contract(fast)
    const int all_large = *large;  // (its wait falls to the staging's)
    __shared__ bf16x8 s_a[4][2][3][64];  // [sample tile][k step][part][lane]: rows of dL/dfeat
    __shared__ bf16x8 s_b[2][3][3][64];  // [sample tile pair][coefficient tile][part][lane]
    __shared__ float4 s_x[64];
    __shared__ float s_par[4][16][17];
    __shared__ int s_big[4];
    const int64_t v = cell_of_block(blockIdx.x, nv);
    const int c = valid[v];
    const int64_t beg = c == 0 ? 0 : prefix[c - 1], end = prefix[c];
    if (beg == end) {
        if (SAMP && threadIdx.x < 192) gsamp[192 * v + threadIdx.x] = 0.0f;
        if (threadIdx.x == 0) cell_large[v] = 0;
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, quad = lane >> 4;
    const float* __restrict__ df = dfeat ? dfeat + 48 * 64 * v : nullptr;
    // First product's k index: lane quarter q holds coefficients 12 q .. 12 q +
    // 11 in slots 0 .. 11 of its 2 x 8; slot 12 of quarter 0 is the density.
    bool big = false;
    for (int i = threadIdx.x; i < 512; i += 256) {
        const int tk = i >> 6, s = 16 * (tk >> 1) + col;
        floatx8 x = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (df) {
            const float* r = df + 48 * s + 12 * quad + 8 * (tk & 1);
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < 4 || (tk & 1) == 0) x[e] = r[e];
        }
        if ((tk & 1) && quad == 0 && ddens) x[4] = ddens[64 * v + s];
        big = big || split_large(make_float4(x[0], x[1], x[2], x[3])) ||
              split_large(make_float4(x[4], x[5], x[6], x[7]));
        bf16x8 p[3];
        split3(x, p);
#pragma unroll
        for (int k = 0; k < 3; k++) s_a[tk >> 1][tk & 1][k][lane] = p[k];
    }
    for (int i = threadIdx.x; i < 384; i += 256) {
        const int hu = i >> 6, h = hu / 3, u = hu % 3;
        floatx8 x = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (df)
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = df[48 * (16 * (2 * h + (e >> 2)) + 4 * quad + (e & 3)) + 16 * u + col];
        bf16x8 p[3];
        split3(x, p);
#pragma unroll
        for (int k = 0; k < 3; k++) s_b[h][u][k][lane] = p[k];
    }
    if (threadIdx.x < 64) {
        const float* x = samples + 3 * (64 * v + threadIdx.x);
        s_x[threadIdx.x] = make_float4(x[0], x[1], x[2], 0.0f);
    }
    const int wave_big = __ballot(big) != 0ull;
    if (lane == 0) s_big[wave] = wave_big;
    __syncthreads();
    const int large_cell = s_big[0] | s_big[1] | s_big[2] | s_big[3];
    if (threadIdx.x == 0) cell_large[v] = (uint8_t)large_cell;
    if (large_cell | all_large) return;  // density_plain_backward_kernel's
    float lf[6];
    if (ADA) density_filter_load(flt, v, lf);
    float dx[SAMP ? 16 : 1][3];
#pragma unroll
    for (int i = 0; i < (SAMP ? 16 : 1); i++) dx[i][0] = dx[i][1] = dx[i][2] = 0.0f;
    const int n = (int)(end - beg);  // a cell lists a Gaussian once: fits 32 bits
    for (int b0 = 16 * wave; b0 < n; b0 += 64) {
        const bool has = b0 + col < n;
        const int g = list[beg + min(b0 + col, n - 1)];
        float4 r0 = rows[3 * (int64_t)g], r1 = rows[3 * (int64_t)g + 1], r2 = rows[3 * (int64_t)g + 2];
        const float4* c4 = reinterpret_cast<const float4*>(sh + 48 * (int64_t)g) + 3 * quad;
        float4 ca = c4[0], cb = c4[1], cc = c4[2];
        // past the list's end: nothing, whatever the last entry is
        if (b0 + 16 > n && !has) r0 = r1 = r2 = ca = cb = cc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        bf16x8 bc[2][3];
        split3(floatx8{ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w}, bc[0]);
        split3(floatx8{cc.x, cc.y, cc.z, cc.w, quad == 0 ? 1.0f : 0.0f, 0.0f, 0.0f, 0.0f}, bc[1]);
        float Q[6] = {r1.x, r1.y, r1.z, r1.w, r2.x, r2.y};
        if (ADA) density_inverse(Q, lf, Q);
        const float o = r0.w;
        // exponent to base 2: e = d^T (-log2(e)/2 Q) d
        constexpr float K2 = -0.72134752044448170f;
        const float q00 = K2 * Q[0], q11 = K2 * Q[1], q22 = K2 * Q[2];
        const float q01 = (SAMP ? 1.0f : 2.0f) * K2 * Q[3], q02 = (SAMP ? 1.0f : 2.0f) * K2 * Q[4],
                    q12 = (SAMP ? 1.0f : 2.0f) * K2 * Q[5];
        // sums over this lane's samples of p = exp(-q/2) da: p, p d, p d d^T
        float sp = 0.0f, s1[3] = {0.0f, 0.0f, 0.0f}, s2[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        floatx4 acc[3];
#pragma unroll
        for (int u = 0; u < 3; u++) acc[u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            floatx8 a;
#pragma unroll
            for (int tt = 0; tt < 2; tt++) {
                const int t = 2 * h + tt;
                // one tile at a time: its LDS operands are not live beside the others'
                __builtin_amdgcn_sched_barrier(0);
                bf16x8 ar[2][3];
#pragma unroll
                for (int k = 0; k < 6; k++) ar[k / 3][k % 3] = s_a[t][k / 3][k % 3][lane];
                floatx4 dh[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
                mfma_split3(ar, bc, dh);
                const floatx4 da = dh[0] + dh[1];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float4 x = s_x[16 * t + 4 * quad + r];
                    const float d0 = x.x - r0.x, d1 = x.y - r0.y, d2 = x.z - r0.z;
                    float e, v0 = 0.0f, v1 = 0.0f, v2 = 0.0f;
                    if (SAMP) {
                        v0 = q00 * d0 + q01 * d1 + q02 * d2;
                        v1 = q01 * d0 + q11 * d1 + q12 * d2;
                        v2 = q02 * d0 + q12 * d1 + q22 * d2;
                        e = v0 * d0 + v1 * d1 + v2 * d2;
                    } else {
                        e = (q00 * d0 + q01 * d1 + q02 * d2) * d0 + (q11 * d1 + q12 * d2) * d1 + q22 * d2 * d2;
                    }
                    const float ex = __builtin_amdgcn_exp2f(e);
                    a[4 * tt + r] = o * ex;
                    const float p = ex * da[r];
                    sp += p;
                    const float p0 = p * d0, p1 = p * d1, p2 = p * d2;
                    s1[0] += p0; s1[1] += p1; s1[2] += p2;
                    s2[0] += p0 * d0; s2[1] += p1 * d1; s2[2] += p2 * d2;
                    s2[3] += p0 * d1; s2[4] += p0 * d2; s2[5] += p1 * d2;
                    if (SAMP) {
                        const float op = o * p;
                        dx[4 * t + r][0] += op * v0;
                        dx[4 * t + r][1] += op * v1;
                        dx[4 * t + r][2] += op * v2;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            bf16x8 ap[3][3], br[3][3];
            split3(a, ap[0]);
#pragma unroll
            for (int k = 0; k < 9; k++) br[k / 3][k % 3] = s_b[h][k / 3][k % 3][lane];
#pragma unroll
            for (int k = 0; k < 3; k++) ap[1][k] = ap[2][k] = ap[0][k];
            mfma_split3(ap, br, acc);
        }
        // the four lanes of a Gaussian
        float sum[10] = {s1[0], s1[1], s1[2], s2[0], s2[1], s2[2], s2[3], s2[4], s2[5], sp};
#pragma unroll
        for (int k = 0; k < 10; k++) {
            sum[k] += __shfl_xor(sum[k], 16);
            sum[k] += __shfl_xor(sum[k], 32);
        }
        // dL/dq = -o p / 2
        const float dq6[6] = {-0.5f * o * sum[3], -0.5f * o * sum[4], -0.5f * o * sum[5],
                              -o * sum[6],        -o * sum[7],        -o * sum[8]};
        float out[10];
        out[0] = o * (Q[0] * sum[0] + Q[3] * sum[1] + Q[4] * sum[2]);
        out[1] = o * (Q[3] * sum[0] + Q[1] * sum[1] + Q[5] * sum[2]);
        out[2] = o * (Q[4] * sum[0] + Q[5] * sum[1] + Q[2] * sum[2]);
        if (ADA) {
            dinv_to_dsigma(Q, dq6, out + 3);
        } else {
#pragma unroll
            for (int k = 0; k < 6; k++) out[3 + k] = dq6[k];
        }
        out[9] = sum[9];
        density_row_add(gacc, g, n - b0, df != nullptr, acc, out, s_par[wave]);
    }
    if (SAMP) {
        // over the 16 lanes of a sample, then over the waves (s_a's space)
        __syncthreads();
        float* s_dx = reinterpret_cast<float*>(s_a);
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int k = 0; k < 3; k++) {
                float w = dx[i][k];
#pragma unroll
                for (int m = 1; m < 16; m <<= 1) w += __shfl_xor(w, m);
                if (col == 0) s_dx[192 * wave + 3 * (16 * (i >> 2) + 4 * quad + (i & 3)) + k] = w;
            }
        __syncthreads();
        if (threadIdx.x < 192) {
            const int i = threadIdx.x;
            // 2 dL/dq Q d = -o p Q d, and the sums hold o p (K2 Q) d
            gsamp[192 * v + i] = 1.3862943611198906f * (s_dx[i] + s_dx[192 + i] + s_dx[384 + i] + s_dx[576 + i]);
        }
    }
}

// The same gradients (but the samples') of a loss whose derivatives are signs,
// sum |feature difference| + w sum |density difference|: one operand of each
// product is exact in one bf16 part, which leaves half of the matrix
// instructions and a third of the operands in LDS. One workgroup takes two
// neighbouring cells (2 p, 2 p + 1), whose lists share most of their Gaussians:
// a Gaussian's row is read, and its sums added to memory, once for both, so
// there are as many atomic requests fewer (they bounded the one-cell form:
// 1M Gaussians on 64^3, 147M pairs, 29.8 -> 19.4 ms, of
// which the 87M merged ones take 17 at 20 G requests a second). Four cells cost
// more in the merge and in idle waves than they saved (30 to 49 ms).
// The lists are in ascending order, so a window of each is merged at a time, up
// to the smaller of the windows' last entries: an entry looks itself up in the
// other window. The merged entries are queued with those of both cells first,
// then those of one alone, and waves take 16 at a time; a cell none of the 16 is
// in is left out, otherwise its share is nothing for those that are not.
template <bool ADA>
__global__ void __launch_bounds__(256, 3) density_sign_backward_kernel(
    int64_t nv, const int* __restrict__ valid, const int64_t* __restrict__ prefix, const int* __restrict__ list,
    const float* __restrict__ samples, const float4* __restrict__ rows, const float* __restrict__ sh,
    DensityFilter flt, const int8_t* __restrict__ signs, float w, float* __restrict__ gacc,
    const uint8_t* __restrict__ skip, const int* __restrict__ large) {
#pragma clang fp contract(fast)
    const int all_large = *large;  // (its wait falls to the staging's)
    constexpr int W = 512;  // entries of a window, two a thread
    __shared__ bf16x8 s_a[2][4][2][64];  // [cell][sample tile][k step][lane]: rows of signs
    __shared__ bf16x8 s_b[2][2][3][64];  // [cell][sample tile pair][coefficient tile][lane]
    __shared__ float4 s_x[2][64];
    __shared__ float s_par[4][16][17];
    __shared__ int s_l[2][W];
    __shared__ int s_q[2 * W];
    __shared__ uint8_t s_in[2 * W];
    __shared__ int s_cnt[3][8];
    __shared__ int s_next;
    // the workgroup of a pair is that of its first valid cell
    const int64_t v0 = cell_of_block(blockIdx.x, nv);
    const int c0 = valid[v0];
    if ((c0 & 1) && v0 > 0 && valid[v0 - 1] == c0 - 1) return;
    const bool two = !(c0 & 1) && v0 + 1 < nv && valid[v0 + 1] == c0 + 1;
    int64_t beg[2];
    int n[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const bool there = (j == 0 || two) && !(skip && skip[v0 + j]);
        beg[j] = !there || c0 + j == 0 ? 0 : prefix[c0 + j - 1];
        n[j] = there ? (int)(prefix[c0 + j] - beg[j]) : 0;  // a cell lists a Gaussian once: fits 32 bits
    }
    if (n[0] + n[1] == 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, quad = lane >> 4;
    // operand layouts as in density_backward_kernel
#pragma unroll
    for (int j = 0; j < 2; j++) {
        if (n[j] == 0) continue;
        const int8_t* sg = signs + DENSITY_SIGNS * 64 * (v0 + j);
        for (int i = threadIdx.x; i < 512; i += 256) {
            const int tk = i >> 6, s = 16 * (tk >> 1) + col;
            const int8_t* r = sg + DENSITY_SIGNS * s + 12 * quad + 8 * (tk & 1);
            floatx8 x = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < 4 || (tk & 1) == 0) x[e] = (float)r[e];
            if ((tk & 1) && quad == 0) x[4] = (float)sg[DENSITY_SIGNS * s + 48];
            s_a[j][tk >> 1][tk & 1][lane] = __builtin_convertvector(x, bf16x8);
        }
        for (int i = threadIdx.x; i < 384; i += 256) {
            const int hu = i >> 6, h = hu / 3, u = hu % 3;
            floatx8 x;
#pragma unroll
            for (int e = 0; e < 8; e++)
                x[e] = (float)sg[DENSITY_SIGNS * (16 * (2 * h + (e >> 2)) + 4 * quad + (e & 3)) + 16 * u + col];
            s_b[j][h][u][lane] = __builtin_convertvector(x, bf16x8);
        }
        if (threadIdx.x < 64) {
            const float* x = samples + 3 * (64 * (v0 + j) + threadIdx.x);
            s_x[j][threadIdx.x] = make_float4(x[0], x[1], x[2], 0.0f);
        }
    }
    if (all_large) return;  // density_plain_backward_kernel's
    float lf[2][6];
    if (ADA) {
        density_filter_load(flt, v0, lf[0]);
        density_filter_load(flt, two ? v0 + 1 : v0, lf[1]);
    }
    int at[2] = {0, 0};
    while (at[0] < n[0] || at[1] < n[1]) {
        // the windows; entries past a list's end sort last
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int i = threadIdx.x + 256 * k;
                s_l[j][i] = i < n[j] - at[j] ? list[beg[j] + at[j] + i] : 0x7fffffff;
            }
        if (threadIdx.x == 0) s_next = 0;
        __syncthreads();
        int limit = 0x7ffffffe;
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (n[j] - at[j] > W) limit = min(limit, s_l[j][W - 1]);
        // this thread's entries: 3 = in both cells, 1 / 2 = in one alone, 0 = not (or the other cell's) to take
        int id[4], in[4], took[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int j = i >> 1;
            id[i] = s_l[j][threadIdx.x + 256 * (i & 1)];
            int lo = 0;  // the last entry of the other window <= id, if any is
#pragma unroll
            for (int step = W / 2; step >= 1; step >>= 1)
                if (s_l[1 - j][lo + step] <= id[i]) lo += step;
            const bool both = s_l[1 - j][lo] == id[i];
            const bool take = id[i] <= limit;
            in[i] = !take ? 0 : both ? (j == 0 ? 3 : 0) : 1 + j;
            took[j] += take ? 1 : 0;
        }
        // places: those of both cells first, then those of the first, of the second
        int cnt[3] = {0, 0, 0}, rank[4];
        const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            rank[i] = 0;
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const uint64_t b = __ballot(in[i] == 3 - m);
                if (in[i] == 3 - m) rank[i] = cnt[m] + __popcll(b & below);
                cnt[m] += __popcll(b);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) took[j] += __shfl_xor(took[j], o);
        if (lane == 0) {
#pragma unroll
            for (int m = 0; m < 3; m++) s_cnt[m][wave] = cnt[m];
            s_cnt[0][4 + wave] = took[0];
            s_cnt[1][4 + wave] = took[1];
        }
        __syncthreads();
        int first[4], total = 0;  // by mark
#pragma unroll
        for (int m = 0; m < 3; m++) {
            first[3 - m] = total;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                first[3 - m] += k < wave ? s_cnt[m][k] : 0;
                total += s_cnt[m][k];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (in[i]) {
                const int q = (in[i] == 3 ? first[3] : in[i] == 2 ? first[2] : first[1]) + rank[i];
                s_q[q] = id[i];
                s_in[q] = (uint8_t)in[i];
            }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            at[0] += s_cnt[0][4 + k];
            at[1] += s_cnt[1][4 + k];
        }
        __syncthreads();
        for (;;) {
            int b0 = 0;
            if (lane == 0) b0 = atomicAdd(&s_next, 16);
            b0 = __builtin_amdgcn_readfirstlane(b0);
            if (b0 >= total) break;
            const int e0 = min(b0 + col, total - 1);
            const int g = s_q[e0], mark = b0 + col < total ? s_in[e0] : 0;
            const float4 r0 = rows[3 * (int64_t)g], r1 = rows[3 * (int64_t)g + 1], r2 = rows[3 * (int64_t)g + 2];
            const float4* c4 = reinterpret_cast<const float4*>(sh + 48 * (int64_t)g) + 3 * quad;
            const float4 ca = c4[0], cb = c4[1], cc = c4[2];
            bf16x8 bc[2][3];
            split3(floatx8{ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w}, bc[0]);
            split3(floatx8{cc.x, cc.y, cc.z, cc.w, quad == 0 ? w : 0.0f, 0.0f, 0.0f, 0.0f}, bc[1]);
            const float o = r0.w;
            float Q[6] = {r1.x, r1.y, r1.z, r1.w, r2.x, r2.y};
            float out[10], sp = 0.0f, s1[3] = {0.0f, 0.0f, 0.0f}, s2[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            if (ADA)
#pragma unroll
                for (int k = 0; k < 10; k++) out[k] = 0.0f;
            // this lane's share of (d mu, d Q or d Sigma, d o): the cell's, added (ADA), or that of both
            const auto add_out = [&](const float Qv[6]) {
                const float dq6[6] = {-0.5f * o * s2[0], -0.5f * o * s2[1], -0.5f * o * s2[2],
                                      -o * s2[3],        -o * s2[4],        -o * s2[5]};
                float v[10];
                v[0] = o * (Qv[0] * s1[0] + Qv[3] * s1[1] + Qv[4] * s1[2]);
                v[1] = o * (Qv[3] * s1[0] + Qv[1] * s1[1] + Qv[5] * s1[2]);
                v[2] = o * (Qv[4] * s1[0] + Qv[5] * s1[1] + Qv[2] * s1[2]);
                if (ADA) {
                    dinv_to_dsigma(Qv, dq6, v + 3);
                } else {
#pragma unroll
                    for (int k = 0; k < 6; k++) v[3 + k] = dq6[k];
                }
                v[9] = sp;
#pragma unroll
                for (int k = 0; k < 10; k++) out[k] = ADA ? out[k] + v[k] : v[k];
            };
            floatx4 acc[3];
#pragma unroll
            for (int u = 0; u < 3; u++) acc[u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int j = 0; j < 2; j++) {
                const bool has = (mark >> j) & 1;
                if (__ballot(has) == 0ull) continue;
                float Qv[6] = {Q[0], Q[1], Q[2], Q[3], Q[4], Q[5]};
                if (ADA) {
                    float l[6];
#pragma unroll
                    for (int k = 0; k < 6; k++) l[k] = j ? lf[1][k] : lf[0][k];
                    density_inverse(Q, l, Qv);
                    // (the other cell's filter may leave a Gaussian that it does not list without an inverse)
#pragma unroll
                    for (int k = 0; k < 6; k++) Qv[k] = has ? Qv[k] : 0.0f;
                    sp = 0.0f;
#pragma unroll
                    for (int k = 0; k < 3; k++) s1[k] = 0.0f;
#pragma unroll
                    for (int k = 0; k < 6; k++) s2[k] = 0.0f;
                }
                // exponent to base 2: e = d^T (-log2(e)/2 Q) d, far below the smallest float where the Gaussian
                // is not of this cell
                constexpr float K2 = -0.72134752044448170f;
                const float none = has ? 0.0f : -16384.0f;
                const float q00 = K2 * Qv[0], q11 = K2 * Qv[1], q22 = K2 * Qv[2];
                const float q01 = 2.0f * K2 * Qv[3], q02 = 2.0f * K2 * Qv[4], q12 = 2.0f * K2 * Qv[5];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    floatx8 a;
#pragma unroll
                    for (int tt = 0; tt < 2; tt++) {
                        const int t = 2 * h + tt;
                        __builtin_amdgcn_sched_barrier(0);
                        floatx4 dh[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
                        const bf16x8 ar[2] = {s_a[j][t][0][lane], s_a[j][t][1][lane]};
#pragma unroll
                        for (int k = 2; k >= 0; k--)
#pragma unroll
                            for (int i = 0; i < 2; i++)
                                dh[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[i], bc[i][k], dh[i], 0, 0, 0);
                        const floatx4 da = dh[0] + dh[1];
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float4 x = s_x[j][16 * t + 4 * quad + r];
                            const float d0 = x.x - r0.x, d1 = x.y - r0.y, d2 = x.z - r0.z;
                            const float e = (q00 * d0 + q01 * d1 + q02 * d2) * d0 + (q11 * d1 + q12 * d2) * d1 +
                                            (q22 * d2 * d2 + none);
                            const float ex = __builtin_amdgcn_exp2f(e);
                            a[4 * tt + r] = o * ex;
                            const float p = ex * da[r];
                            sp += p;
                            const float p0 = p * d0, p1 = p * d1, p2 = p * d2;
                            s1[0] += p0; s1[1] += p1; s1[2] += p2;
                            s2[0] += p0 * d0; s2[1] += p1 * d1; s2[2] += p2 * d2;
                            s2[3] += p0 * d1; s2[4] += p0 * d2; s2[5] += p1 * d2;
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    bf16x8 ap[3], br[3];
                    split3(a, ap);
#pragma unroll
                    for (int u = 0; u < 3; u++) br[u] = s_b[j][h][u][lane];
#pragma unroll
                    for (int k = 2; k >= 0; k--)
#pragma unroll
                        for (int u = 0; u < 3; u++)
                            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[k], br[u], acc[u], 0, 0, 0);
                }
                if (ADA) add_out(Qv);
            }
            if (!ADA) add_out(Q);
#pragma unroll
            for (int k = 0; k < 10; k++) {
                out[k] += __shfl_xor(out[k], 16);
                out[k] += __shfl_xor(out[k], 32);
            }
            density_row_add(gacc, g, total - b0, true, acc, out, s_par[wave]);
        }
        __syncthreads();
    }
}

// The gradients of both kernels above with operands from SPLIT_MOST on, infinities
// among them: plain FP32 sums, of all cells where *large, else (cell_large not
// null) of those marked. One wave a cell, each lane with the next Gaussian of its
// list, and 64 cells looked at at a time: without any, as good as always, it
// takes 4 us. SIGN: the output gradients are signs (density_sign_backward_kernel).
template <bool SIGN>
__global__ void __launch_bounds__(64) density_plain_backward_kernel(
    int64_t nv, const int* __restrict__ valid, const int64_t* __restrict__ prefix, const int* __restrict__ list,
    const float* __restrict__ samples, const float4* __restrict__ rows, const float* __restrict__ sh,
    DensityFilter flt, const float* __restrict__ dfeat, const float* __restrict__ ddens,
    const int8_t* __restrict__ signs, float w, float* __restrict__ gsamp, float* __restrict__ gacc,
    const uint8_t* __restrict__ skip, const int* __restrict__ large, const uint8_t* __restrict__ cell_large) {
#pragma clang fp contract(fast)
    __shared__ float s_x[64][3], s_df[64][49], s_dx[64][3];
    const int lane = threadIdx.x;
    const bool every = *large != 0;
    for (int64_t v0 = 64 * (int64_t)blockIdx.x; v0 < nv; v0 += 64 * (int64_t)gridDim.x) {
        const int64_t mine = v0 + lane;
        const bool take = mine < nv && (every || (cell_large && cell_large[mine])) && !(skip && skip[mine]);
        for (uint64_t left = __ballot(take); left != 0ull; left &= left - 1ull) {
            const int64_t v = v0 + __builtin_ctzll(left), at = 64 * v + lane;
            const int c = valid[v];
            const int64_t beg = c == 0 ? 0 : prefix[c - 1], end = prefix[c];
            __syncthreads();
            for (int k = 0; k < 3; k++) {
                s_x[lane][k] = samples[3 * at + k];
                s_dx[lane][k] = 0.0f;
            }
            if (SIGN) {
                const int8_t* sg = signs + DENSITY_SIGNS * at;
                for (int k = 0; k < 48; k++) s_df[lane][k] = (float)sg[k];
                s_df[lane][48] = sg[48] > 0 ? w : sg[48] < 0 ? -w : 0.0f;
            } else {
                for (int k = 0; k < 48; k++) s_df[lane][k] = dfeat ? dfeat[48 * at + k] : 0.0f;
                s_df[lane][48] = ddens ? ddens[at] : 0.0f;
            }
            __syncthreads();
            float lf[6];
            if (flt.ada) density_filter_load(flt, v, lf);
            for (int64_t b0 = beg; b0 < end; b0 += 64) {
                const bool has = b0 + lane < end;
                const int64_t g = has ? list[b0 + lane] : 0;
                float mu[3] = {0.0f, 0.0f, 0.0f}, o = 0.0f, Q[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                float cg[48], gc[48], gmu[3] = {0.0f, 0.0f, 0.0f}, gQ[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, go = 0.0f;
                if (has) {
                    const float4 r0 = rows[3 * g], r1 = rows[3 * g + 1], r2 = rows[3 * g + 2];
                    mu[0] = r0.x; mu[1] = r0.y; mu[2] = r0.z; o = r0.w;
                    Q[0] = r1.x; Q[1] = r1.y; Q[2] = r1.z; Q[3] = r1.w; Q[4] = r2.x; Q[5] = r2.y;
                    if (flt.ada) density_inverse(Q, lf, Q);
                }
#pragma unroll
                for (int k = 0; k < 48; k++) {
                    cg[k] = has ? sh[48 * g + k] : 0.0f;
                    gc[k] = 0.0f;
                }
                for (int s = 0; s < 64; s++) {
                    const float d0 = s_x[s][0] - mu[0], d1 = s_x[s][1] - mu[1], d2 = s_x[s][2] - mu[2];
                    const float e0 = Q[0] * d0 + Q[3] * d1 + Q[4] * d2, e1 = Q[3] * d0 + Q[1] * d1 + Q[5] * d2,
                                e2 = Q[4] * d0 + Q[5] * d1 + Q[2] * d2;
                    const float ex = __expf(-0.5f * (e0 * d0 + e1 * d1 + e2 * d2)), a = o * ex;
                    float da = s_df[s][48];
#pragma unroll
                    for (int k = 0; k < 48; k++) {
                        da += s_df[s][k] * cg[k];
                        gc[k] += a * s_df[s][k];
                    }
                    go += ex * da;
                    const float dq = -0.5f * a * da;  // dL/dq
                    gQ[0] += dq * d0 * d0; gQ[1] += dq * d1 * d1; gQ[2] += dq * d2 * d2;
                    gQ[3] += 2.0f * dq * d0 * d1; gQ[4] += 2.0f * dq * d0 * d2; gQ[5] += 2.0f * dq * d1 * d2;
                    float x[3] = {2.0f * dq * e0, 2.0f * dq * e1, 2.0f * dq * e2};
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        gmu[k] -= x[k];
                        for (int m = 32; m > 0; m >>= 1) x[k] += __shfl_xor(x[k], m);
                        if (lane == 0) s_dx[s][k] += x[k];
                    }
                }
                if (!has) continue;
                if (flt.ada) {
                    const float dq6[6] = {gQ[0], gQ[1], gQ[2], gQ[3], gQ[4], gQ[5]};
                    dinv_to_dsigma(Q, dq6, gQ);
                }
                float* row = gacc + 64 * g;
#pragma unroll
                for (int k = 0; k < 48; k++) unsafeAtomicAdd(row + k, gc[k]);
#pragma unroll
                for (int k = 0; k < 3; k++) unsafeAtomicAdd(row + 48 + k, gmu[k]);
#pragma unroll
                for (int k = 0; k < 6; k++) unsafeAtomicAdd(row + 51 + k, gQ[k]);
                unsafeAtomicAdd(row + 57, go);
            }
            __syncthreads();
            if (gsamp)
                for (int k = 0; k < 3; k++) gsamp[3 * at + k] = s_dx[lane][k];
        }
    }
}

// dL/dSigma of a density Gaussian (packed as dinv_to_dsigma writes it) back to
// its rotation q (unnormalised, as stored) and scale s, Sigma = R(q/|q|)
// diag(s^2) R^T + L. Adds into dq and ds.
__device__ __forceinline__ void density_sigma_backward(const float* __restrict__ rot,
                                                       const float* __restrict__ scale, int64_t g, const float ds6[6],
                                                       float dq[4], float ds[3]) {
    const float s1[3] = {scale[3 * g], scale[3 * g + 1], scale[3 * g + 2]};
    const float q1[4] = {rot[4 * g], rot[4 * g + 1], rot[4 * g + 2], rot[4 * g + 3]};
    float qn[4] = {q1[0], q1[1], q1[2], q1[3]};
    quat_normalize(qn);
    float R[3][3];
    quat_to_mat(qn[0], qn[1], qn[2], qn[3], R);
    const float dS[3][3] = {{ds6[0], 0.5f * ds6[3], 0.5f * ds6[4]},
                            {0.5f * ds6[3], ds6[1], 0.5f * ds6[5]},
                            {0.5f * ds6[4], 0.5f * ds6[5], ds6[2]}};
    float dR[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < 3; j++) acc += (dS[a][j] + dS[j][a]) * R[j][b];
            dR[a][b] = s1[b] * s1[b] * acc;
        }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float dD = 0.0f;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) dD += dS[i][j] * R[i][k] * R[j][k];
        ds[k] += dD * 2.0f * s1[k];
    }
    float dqn[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    quat_to_mat_backward(qn, dR, dqn);
    quat_normalize_backward(q1, dqn, dq);
}

// The accumulated covariance gradient d6 (d[3..8] of the density backward) of
// Gaussian g back to (q, s): dL/dQ with the scalar filter (Sigma = R diag(s^2)
// R^T + lpf I, dSigma = -Q dQ Q), dL/dSigma itself with an adaptive one.
__device__ __forceinline__ void density_cov_backward(const float* __restrict__ rot, const float* __restrict__ scale,
                                                     int64_t g, const DensityFilter& flt, const float d6[6],
                                                     float dq[4], float ds[3]) {
    float ds6[6];
    if (flt.ada) {
#pragma unroll
        for (int k = 0; k < 6; k++) ds6[k] = d6[k];
    } else {
        float S[6], L[6], Qv[6];
        density_cov(rot, scale, g, S);
        density_filter_load(flt, 0, L);
        density_inverse(S, L, Qv);
        dinv_to_dsigma(Qv, d6, ds6);
    }
    density_sigma_backward(rot, scale, g, ds6, dq, ds);
}

// The density gradients of every Gaussian's own attributes but the SH (the VJP
// of the density sample, arapgs_density_backward): position, rotation (as
// stored), scale and opacity from the accumulator rows, and the SH copied out of
// them where dsh is given.
__global__ void __launch_bounds__(256) density_attr_grad_kernel(int64_t N, const float* __restrict__ rot,
                                                                const float* __restrict__ scale,
                                                                const float* __restrict__ gacc, DensityFilter flt,
                                                                float* __restrict__ dsh, float* __restrict__ dpos, float* __restrict__ drot,
                                                                float* __restrict__ dscale,
                                                                float* __restrict__ dopac) {
    const int64_t g0 = (int64_t)blockIdx.x * blockDim.x, g = g0 + threadIdx.x;
    if (dsh) {
        const int n = 48 * (int)min<int64_t>(blockDim.x, N - g0);
        for (int i = threadIdx.x; i < n; i += blockDim.x) dsh[48 * g0 + i] = gacc[64 * (g0 + i / 48) + i % 48];
    }
    if (g >= N) return;
    const float4* r = reinterpret_cast<const float4*>(gacc + 64 * g + 48);
    const float4 a = r[0], b = r[1], c = r[2];
    const float d6[6] = {a.w, b.x, b.y, b.z, b.w, c.x};
    float dq[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ds[3] = {0.0f, 0.0f, 0.0f};
    density_cov_backward(rot, scale, g, flt, d6, dq, ds);
    dpos[3 * g] = a.x; dpos[3 * g + 1] = a.y; dpos[3 * g + 2] = a.z;
#pragma unroll
    for (int k = 0; k < 4; k++) drot[4 * g + k] = dq[k];
#pragma unroll
    for (int k = 0; k < 3; k++) dscale[3 * g + k] = ds[k];
    dopac[g] = c.y;
}

// One thread per Gaussian: the adjoint of everything between the rest
// attributes and (mu', q', s', c'). gr: the renderer's per-Gaussian gradient
// (d mu' 3, d q' 4, d s' 3, d c' 48); gacc: the density's (rows of 64,
// density_backward_kernel) or null; opacities are constants here. Writes d e' (18) and d q0, d s0.
__global__ void __launch_bounds__(128) six_point_backward_kernel(
    int64_t N, int K, const NodeXf* __restrict__ table, const uint32_t* __restrict__ ends_idx,
    const float* __restrict__ ends_w, const float* __restrict__ ends, const float* __restrict__ rot0,
    const float* __restrict__ scale0, const float* __restrict__ sh0, const float* __restrict__ rot1,
    const float* __restrict__ scale1, const float* __restrict__ gr, const float* __restrict__ gacc, DensityFilter flt, float pad, float coeff, const ShRotTables* __restrict__ Tsh, float* __restrict__ gends,
    float* __restrict__ drot0, float* __restrict__ dscale0) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= N) return;
    const float* r = gr + 58 * g;
    float dmu[3] = {r[0], r[1], r[2]};
    float dq1[4] = {r[3], r[4], r[5], r[6]};
    float ds1[3] = {r[7], r[8], r[9]};
    float dc1[48];
#pragma unroll
    for (int k = 0; k < 48; k++) dc1[k] = r[10 + k];
    if (gacc) {
        const float4* r4 = reinterpret_cast<const float4*>(gacc + 64 * g + 48);
        const float4 a = r4[0], b = r4[1], c = r4[2];
        const float d6[6] = {a.w, b.x, b.y, b.z, b.w, c.x};
        dmu[0] += a.x; dmu[1] += a.y; dmu[2] += a.z;
        const float4* d4 = reinterpret_cast<const float4*>(gacc + 64 * g);
#pragma unroll
        for (int k = 0; k < 12; k++) {
            const float4 v = d4[k];
            dc1[4 * k] += v.x; dc1[4 * k + 1] += v.y; dc1[4 * k + 2] += v.z; dc1[4 * k + 3] += v.w;
        }
        density_cov_backward(rot1, scale1, g, flt, d6, dq1, ds1);
    }

    // recompute the six-point forward from the blended end points
    float e[6][3];
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
        for (int c = 0; c < 3; c++) e[p][c] = ends[18 * g + 3 * p + c];
    double M[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int c = 0; c < 3; c++) M[c][i] = 0.5 * ((double)e[2 * i][c] - (double)e[2 * i + 1][c]);
    double Rd[3][3], Vd[3][3], sig[3];
    polar3_fp64_svd(M, Rd, Vd, sig);
    double Sd[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
        Sd[i] = Vd[i][0] * sig[0] * Vd[i][0] + Vd[i][1] * sig[1] * Vd[i][1] + Vd[i][2] * sig[2] * Vd[i][2];
    float Rf[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) Rf[i][j] = (float)Rd[i][j];
    float qm[4];
    mat_to_quat(Rf, qm);
    float q[4] = {qm[0], qm[1], qm[2], qm[3]};
    quat_normalize(q);

    // SH: c' = rot(R(normalise(q qi))) c0, qi = conj(q0) / |q0|^2
    const float qo[4] = {rot0[4 * g], rot0[4 * g + 1], rot0[4 * g + 2], rot0[4 * g + 3]};
    const float n2 = qo[0] * qo[0] + qo[1] * qo[1] + qo[2] * qo[2] + qo[3] * qo[3];
    const float qi[4] = {qo[0] / n2, -qo[1] / n2, -qo[2] / n2, -qo[3] / n2};
    float qm2[4];
    quat_mul(q, qi, qm2);
    float qr[4] = {qm2[0], qm2[1], qm2[2], qm2[3]};
    quat_normalize(qr);
    float Rr[3][3];
    quat_to_mat(qr[0], qr[1], qr[2], qr[3], Rr);
    float c0[48];
    const float4* c4 = reinterpret_cast<const float4*>(sh0 + 48 * g);
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const float4 v = c4[k];
        c0[4 * k] = v.x; c0[4 * k + 1] = v.y; c0[4 * k + 2] = v.z; c0[4 * k + 3] = v.w;
    }
    float dRr[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    sh_rotate_backward(*Tsh, Rr, c0, dc1, dRr);
    float dqr[4] = {0.0f, 0.0f, 0.0f, 0.0f}, dqm2[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    quat_to_mat_backward(qr, dRr, dqr);
    quat_normalize_backward(qm2, dqr, dqm2);
    float dqi[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    quat_mul_backward(q, qi, dqm2, dq1, dqi);
    // qi_k = c_k qo_k / n2 (c = 1, -1, -1, -1)
    const float cs[4] = {1.0f, -1.0f, -1.0f, -1.0f};
    float dq0[4];
    {
        float sdot = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) sdot += dqi[k] * cs[k] * qo[k];
#pragma unroll
        for (int k = 0; k < 4; k++) dq0[k] = cs[k] * dqi[k] / n2 - 2.0f * qo[k] * sdot / (n2 * n2);
    }

    // scales: s'_i = S_ii / ((s0_i + pad) coeff) s0_i
    double dSd[3];
    float ds0[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const float s0 = scale0[3 * g + i];
        const float den = (s0 + pad) * coeff;
        dSd[i] = (double)(ds1[i] * s0 / den);
        ds0[i] = ds1[i] * (float)Sd[i] * pad / (coeff * (s0 + pad) * (s0 + pad));
    }
    // q' = normalise(mat_to_quat(R))
    float dqm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    quat_normalize_backward(qm, dq1, dqm);
    float dRf[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    mat_to_quat_backward(Rf, dqm, dRf);
    double dRd[3][3], dM[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) dRd[i][j] = (double)dRf[i][j];
    polar3_fp64_backward(Rd, Vd, sig, dRd, dSd, dM);

    // d e' from M and from the centre
    float de[6][3];
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
        for (int c = 0; c < 3; c++) de[p][c] = dmu[c] / 6.0f;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float h = (float)(0.5 * dM[c][i]);
            de[2 * i][c] += h;
            de[2 * i + 1][c] -= h;
        }
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
        for (int c = 0; c < 3; c++) gends[18 * g + 3 * p + c] = de[p][c];

    // blend adjoint to the rest end points: d e = sum_j w_j R_j^T d e'
    float dE[6][3];
#pragma unroll
    for (int p = 0; p < 6; p++) {
        dE[p][0] = dE[p][1] = dE[p][2] = 0.0f;
        const int64_t pt = 6 * g + p;
        for (int j = 0; j < K; j++) {
            const NodeXf& nd = table[ends_idx[pt * K + j]];
            const float w = ends_w[pt * K + j];
#pragma unroll
            for (int c = 0; c < 3; c++)
                dE[p][c] += w * (nd.R[c] * de[p][0] + nd.R[3 + c] * de[p][1] + nd.R[6 + c] * de[p][2]);
        }
    }
    // end points: e_{i+-} = mu0 +- R0[:, i] (s0_i + pad) coeff, R0 = R(q0 / |q0|)
    float qn0[4] = {qo[0], qo[1], qo[2], qo[3]};
    quat_normalize(qn0);
    float R0[3][3];
    quat_to_mat(qn0[0], qn0[1], qn0[2], qn0[3], R0);
    float dR0[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const float len = (scale0[3 * g + i] + pad) * coeff;
        float dlen = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float dd = dE[2 * i][c] - dE[2 * i + 1][c];
            dlen += R0[c][i] * dd;
            dR0[c][i] = len * dd;
        }
        ds0[i] += dlen * coeff;
    }
    float dqn0[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    quat_to_mat_backward(qn0, dR0, dqn0);
    quat_normalize_backward(qo, dqn0, dq0);
#pragma unroll
    for (int k = 0; k < 4; k++) drot0[4 * g + k] = dq0[k];
#pragma unroll
    for (int k = 0; k < 3; k++) dscale0[3 * g + k] = ds0[k];
}

// Entry e of the inverse index is (point, slot) = (e / K, e % K) over the
// 6N end points followed by the S samples; its node is the blend id.
__global__ void entry_keys_kernel(int64_t n_end_entries, int64_t n_entries, const uint32_t* __restrict__ ends_idx,
                                  const uint32_t* __restrict__ sample_idx, uint64_t* __restrict__ keys,
                                  uint32_t* __restrict__ vals) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_entries) return;
    keys[e] = e < n_end_entries ? ends_idx[e] : sample_idx[e - n_end_entries];
    vals[e] = (uint32_t)e;
}

__global__ void zero_u32_kernel(uint32_t* __restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

__global__ void node_ranges_kernel(const uint64_t* __restrict__ keys, int64_t n, int M, uint2* __restrict__ rng) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = (uint32_t)keys[i];
    if (k >= (uint32_t)M) return;  // not a node id: dropped
    if (i == 0 || (uint32_t)keys[i - 1] != k) rng[k].x = (uint32_t)i;
    if (i == n - 1 || (uint32_t)keys[i + 1] != k) rng[k].y = (uint32_t)(i + 1);
}

// d R_j = sum w d e' (p - g_j)^T and d t_j = sum w d e' over the node's
// entries (p the blend input: rest end point or rest sample). Thread partials
// in FP64, fixed-order block reduction: deterministic.
__global__ void __launch_bounds__(256) node_gather_kernel(int M, int K, int64_t n_end_entries,
                                                          const uint2* __restrict__ rng,
                                                          const uint32_t* __restrict__ entries,
                                                          const NodeXf* __restrict__ table,
                                                          const float* __restrict__ ends_w,
                                                          const float* __restrict__ ends0,
                                                          const float* __restrict__ gends,
                                                          const float* __restrict__ sample_w,
                                                          const float* __restrict__ samples0,
                                                          const float* __restrict__ gsamp,
                                                          NodeXf* __restrict__ dtable) {
    __shared__ double s_red[4][12];
    const int n = blockIdx.x;
    if (n >= M) return;
    const uint2 r = rng[n];
    const float gx = table[n].g[0], gy = table[n].g[1], gz = table[n].g[2];
    double acc[12];
#pragma unroll
    for (int k = 0; k < 12; k++) acc[k] = 0.0;
    for (uint32_t i = r.x + threadIdx.x; i < r.y; i += blockDim.x) {
        const uint32_t e = entries[i];
        float w, px, py, pz, d0, d1, d2;
        if ((int64_t)e < n_end_entries) {
            const uint32_t p = e / (uint32_t)K;
            w = ends_w[e];
            px = ends0[3 * (int64_t)p]; py = ends0[3 * (int64_t)p + 1]; pz = ends0[3 * (int64_t)p + 2];
            d0 = gends[3 * (int64_t)p]; d1 = gends[3 * (int64_t)p + 1]; d2 = gends[3 * (int64_t)p + 2];
        } else {
            const int64_t es = (int64_t)e - n_end_entries;
            const int64_t s = es / K;
            w = sample_w[es];
            px = samples0[3 * s]; py = samples0[3 * s + 1]; pz = samples0[3 * s + 2];
            d0 = gsamp[3 * s]; d1 = gsamp[3 * s + 1]; d2 = gsamp[3 * s + 2];
        }
        const double tx = (double)(px - gx), ty = (double)(py - gy), tz = (double)(pz - gz);
        const double wd0 = (double)w * d0, wd1 = (double)w * d1, wd2 = (double)w * d2;
        acc[0] += wd0 * tx; acc[1] += wd0 * ty; acc[2] += wd0 * tz;
        acc[3] += wd1 * tx; acc[4] += wd1 * ty; acc[5] += wd1 * tz;
        acc[6] += wd2 * tx; acc[7] += wd2 * ty; acc[8] += wd2 * tz;
        acc[9] += wd0; acc[10] += wd1; acc[11] += wd2;
    }
#pragma unroll
    for (int k = 0; k < 12; k++) {
        double v = acc[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        acc[k] = v;
    }
    const int wid = threadIdx.x >> 6, wl = threadIdx.x & 63;
    if (wl == 0)
#pragma unroll
        for (int k = 0; k < 12; k++) s_red[wid][k] = acc[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        const int k = threadIdx.x;
        const float v = (float)(s_red[0][k] + s_red[1][k] + s_red[2][k] + s_red[3][k]);
        float* o = reinterpret_cast<float*>(dtable + n);
        if (k < 9) o[3 + k] = v;   // R, row-major
        else o[12 + (k - 9)] = v;  // t
    }
    if (threadIdx.x >= 12 && threadIdx.x < 16) {
        float* o = reinterpret_cast<float*>(dtable + n);
        const int k = threadIdx.x - 12;  // g (3) and pad: not differentiated
        o[k < 3 ? k : 15] = 0.0f;
    }
}

// ---------------------------------------------------------------- realignment
// raw parameters -> activated: s = exp(log s), o = sigmoid(logit o)
__global__ void __launch_bounds__(256) activate_kernel(int64_t N, const float* __restrict__ log_scale,
                                                       const float* __restrict__ logit_opac, float* __restrict__ scale,
                                                       float* __restrict__ opac) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= N) return;
#pragma unroll
    for (int k = 0; k < 3; k++) scale[3 * g + k] = expf(log_scale[3 * g + k]);
    opac[g] = 1.0f / (1.0f + expf(-logit_opac[g]));
}

// Cells whose lists hold no moved Gaussian (the reference's current static
// grids, GaussianView.cpp:3850-3852): one wave per valid cell.
__global__ void __launch_bounds__(64) static_cells_kernel(int64_t nv, const int* __restrict__ valid,
                                                          const int64_t* __restrict__ prefix,
                                                          const int* __restrict__ list,
                                                          const uint8_t* __restrict__ moved,
                                                          uint8_t* __restrict__ stat) {
    const int64_t v = blockIdx.x;
    if (v >= nv) return;
    const int c = valid[v];
    const int64_t beg = c == 0 ? 0 : prefix[c - 1], end = prefix[c];
    bool any = false;
    for (int64_t i = beg + threadIdx.x; i < end && !any; i += 64) any = moved[list[i]] != 0;
    any = __ballot(any) != 0ull;
    if (threadIdx.x == 0) stat[v] = any ? 0 : 1;
}

// Per-cell convergence of the realignment: the first step of a run (a new
// realignment or new options) records every cell's loss and clears the
// converged flags; a later step marks a cell converged once its loss is at
// most tol times that record (sticky, also across re-binnings, as the
// reference's grid_is_converged). skip = static or converged.
__global__ void __launch_bounds__(256) converge_kernel(int64_t nv, const float* __restrict__ cell_loss,
                                                       float* __restrict__ cell_ref,
                                                       const uint8_t* __restrict__ stat, float tol, int first,
                                                       uint8_t* __restrict__ conv, uint8_t* __restrict__ skip) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const bool st = stat && stat[v];
    if (first) {
        cell_ref[v] = cell_loss[v];
        conv[v] = 0;
        skip[v] = st ? 1 : 0;
        return;
    }
    const bool c = conv[v] || (tol > 0.0f && cell_loss[v] <= tol * cell_ref[v]);
    conv[v] = c ? 1 : 0;
    skip[v] = (st || c) ? 1 : 0;
}

// ExpandOpRange (GaussianView.cpp:4320-4360): every cell that is, or is a face
// neighbour (clamped to the grid) of, a non-converged valid cell is marked in
// map (G^3 bytes, cleared by the caller) ...
__global__ void __launch_bounds__(256) expand_mark_kernel(int64_t nv, const int* __restrict__ valid,
                                                          const uint8_t* __restrict__ conv, int G,
                                                          uint8_t* __restrict__ map) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv || conv[v]) return;
    const int c = valid[v];
    const int z = c % G, y = (c / G) % G, x = c / (G * G);
    const int64_t GG = (int64_t)G * G;
    map[c] = 1;
    map[(int64_t)max(x - 1, 0) * GG + (int64_t)y * G + z] = 1;
    map[(int64_t)min(x + 1, G - 1) * GG + (int64_t)y * G + z] = 1;
    map[(int64_t)x * GG + (int64_t)max(y - 1, 0) * G + z] = 1;
    map[(int64_t)x * GG + (int64_t)min(y + 1, G - 1) * G + z] = 1;
    map[(int64_t)x * GG + (int64_t)y * G + max(z - 1, 0)] = 1;
    map[(int64_t)x * GG + (int64_t)y * G + min(z + 1, G - 1)] = 1;
}

// ... and every marked valid cell is no longer converged.
__global__ void __launch_bounds__(256) expand_apply_kernel(int64_t nv, const int* __restrict__ valid,
                                                           const uint8_t* __restrict__ map,
                                                           const uint8_t* __restrict__ stat,
                                                           uint8_t* __restrict__ conv, uint8_t* __restrict__ skip) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv || !map[valid[v]]) return;
    conv[v] = 0;
    skip[v] = (stat && stat[v]) ? 1 : 0;
}

// One Adam step per Gaussian over its 59 raw parameters (pos 3, rot 4,
// log-scale 3, logit-opacity 1, SH 48); the activated gradients are chained to
// the raw ones (d log s = d s * s, d logit o = d o * o (1 - o)); dsh lies in the
// first 48 of rows of 64 (density_backward_kernel's). m and v are
// component-major (k * N + g); bc1 / bc2 are the bias corrections 1 - beta^t.
__global__ void __launch_bounds__(256) adam_kernel(int64_t N, const float* __restrict__ dpos,
                                                   const float* __restrict__ drot, const float* __restrict__ dscale,
                                                   const float* __restrict__ dopac, const float* __restrict__ dsh,
                                                   const float* __restrict__ scale, const float* __restrict__ opac,
                                                   float* __restrict__ pos, float* __restrict__ rot,
                                                   float* __restrict__ log_scale, float* __restrict__ logit_opac,
                                                   float* __restrict__ sh, float* __restrict__ m, float* __restrict__ v,
                                                   float lr_pos, float lr_rot, float lr_scale, float lr_opac,
                                                   float lr_sh, float b1, float b2, float eps, float bc1, float bc2,
                                                   const uint8_t* __restrict__ moved,
                                                   const float* __restrict__ max_scale) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= N) return;
    if (moved && !moved[g]) return;  // "Only Optimize Deformed Region": the rest stays as it is
    auto step = [&](int k, float grad, float lr, float& p) {
        float& mk = m[k * N + g];
        float& vk = v[k * N + g];
        mk = b1 * mk + (1.0f - b1) * grad;
        vk = b2 * vk + (1.0f - b2) * grad * grad;
        p -= lr * (mk / bc1) / (sqrtf(vk / bc2) + eps);
    };
#pragma unroll
    for (int c = 0; c < 3; c++) step(c, dpos[3 * g + c], lr_pos, pos[3 * g + c]);
#pragma unroll
    for (int c = 0; c < 4; c++) step(3 + c, drot[4 * g + c], lr_rot, rot[4 * g + c]);
#pragma unroll
    for (int c = 0; c < 3; c++) step(7 + c, dscale[3 * g + c] * scale[3 * g + c], lr_scale, log_scale[3 * g + c]);
    const float o = opac[g];
    step(10, dopac[g] * o * (1.0f - o), lr_opac, logit_opac[g]);
#pragma unroll 4
    for (int c = 0; c < 48; c++) step(11 + c, dsh[64 * g + c], lr_sh, sh[48 * g + c]);
    if (max_scale)
#pragma unroll
        for (int c = 0; c < 3; c++) log_scale[3 * g + c] = fminf(log_scale[3 * g + c], logf(max_scale[3 * g + c]));
}

}  // namespace

int launch_activate(int64_t N, const float* log_scale, const float* logit_opac, float* scale, float* opac,
                    hipStream_t st) {
    if (N <= 0) return 0;
    hipLaunchKernelGGL(activate_kernel, dim3(nblk(N, 256)), dim3(256), 0, st, N, log_scale, logit_opac, scale, opac);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_static_cells(int64_t nv, const int* valid, const int64_t* prefix, const int* list, const uint8_t* moved,
                        uint8_t* stat, hipStream_t st) {
    if (nv <= 0) return 0;
    hipLaunchKernelGGL(static_cells_kernel, dim3((unsigned)nv), dim3(64), 0, st, nv, valid, prefix, list, moved, stat);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_converge(int64_t nv, const float* cell_loss, float* cell_ref, const uint8_t* stat, float tol, int first,
                    uint8_t* conv, uint8_t* skip, hipStream_t st) {
    if (nv <= 0) return 0;
    hipLaunchKernelGGL(converge_kernel, dim3(nblk(nv, 256)), dim3(256), 0, st, nv, cell_loss, cell_ref, stat, tol,
                       first, conv, skip);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_expand_op_range(int64_t nv, const int* valid, int G, const uint8_t* stat, uint8_t* conv, uint8_t* skip,
                           uint8_t* map, hipStream_t st) {
    if (nv <= 0) return 0;
    const int64_t gc = (int64_t)G * G * G;
    hipLaunchKernelGGL(zero_f32_kernel, dim3(std::min<int64_t>(nblk((gc + 3) / 4, 256), 4096)), dim3(256), 0, st,
                       reinterpret_cast<float*>(map), (gc + 3) / 4);
    hipLaunchKernelGGL(expand_mark_kernel, dim3(nblk(nv, 256)), dim3(256), 0, st, nv, valid, conv, G, map);
    hipLaunchKernelGGL(expand_apply_kernel, dim3(nblk(nv, 256)), dim3(256), 0, st, nv, valid, map, stat, conv, skip);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_adam(int64_t N, const float* dpos, const float* drot, const float* dscale, const float* dopac,
                const float* dsh, const float* scale, const float* opac, float* pos, float* rot, float* log_scale,
                float* logit_opac, float* sh, float* m, float* v, const float lr[5], float b1, float b2, float eps,
                float bc1, float bc2, const uint8_t* moved, const float* max_scale, hipStream_t st) {
    if (N <= 0) return 0;
    hipLaunchKernelGGL(adam_kernel, dim3(nblk(N, 256)), dim3(256), 0, st, N, dpos, drot, dscale, dopac, dsh, scale,
                       opac, pos, rot, log_scale, logit_opac, sh, m, v, lr[0], lr[1], lr[2], lr[3], lr[4], b1, b2, eps,
                       bc1, bc2, moved, max_scale);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_zero_f32(float* p, int64_t n, hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(zero_f32_kernel, dim3(std::min<unsigned>(nblk(n, 256), 8192)), dim3(256), 0, st, p, n);
    HIP_RET(hipGetLastError());
    return 0;
}

namespace {
// accumulators (DENSITY_ACC floats a Gaussian), the word that says that an operand is large, parameter rows and
// the cells' marks
struct DensityWs {
    float* acc;
    int* large;
    float4* rows;
    uint8_t* cell_large;
    DensityWs(float* ws, int64_t n) : acc(ws) {
        large = reinterpret_cast<int*>(ws + DENSITY_ACC * n);
        rows = reinterpret_cast<float4*>(ws + DENSITY_ACC * n + 4);
        cell_large = reinterpret_cast<uint8_t*>(ws + (DENSITY_ACC + 12) * n + 4);
    }
};
}  // namespace

size_t density_ws_floats(int64_t n_gauss, int64_t nv) {
    return (size_t)((DENSITY_ACC + 12) * std::max<int64_t>(n_gauss, 1) + 4 + (nv + 3) / 4);
}

int launch_density_ws_clear(int64_t n_gauss, float* ws, hipStream_t st) {
    return launch_zero_f32(ws, DENSITY_ACC * n_gauss + 4, st);
}

int launch_density_backward(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                            const float* samples, const float* pos, const float* rot, const float* scale,
                            const float* opacity, const float* sh, DensityFilter flt, const float* dfeat,
                            const float* ddens, float* gsamp, float* ws, hipStream_t st) {
    if (nv <= 0 || n_gauss <= 0) return 0;
    const DensityWs W(ws, n_gauss);
    hipLaunchKernelGGL(density_rows_kernel, dim3(nblk(n_gauss, 256)), dim3(256), 0, st, n_gauss, pos, rot, scale,
                       opacity, sh, flt, W.rows, W.large);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nv), dim3(256), 0, st, nv, valid, prefix, list, samples,
                           (const float4*)W.rows, sh, flt, dfeat, ddens, gsamp, W.acc, (const int*)W.large, W.cell_large);
    };
    if (flt.ada && gsamp) launch(density_backward_kernel<true, true>);
    else if (flt.ada) launch(density_backward_kernel<true, false>);
    else if (gsamp) launch(density_backward_kernel<false, true>);
    else launch(density_backward_kernel<false, false>);
    hipLaunchKernelGGL(density_plain_backward_kernel<false>, dim3(std::min(nblk(nv, 64), 4096u)), dim3(64), 0, st, nv,
                       valid, prefix, list, samples, (const float4*)W.rows, sh, flt, dfeat, ddens,
                       (const int8_t*)nullptr, 0.0f, gsamp, W.acc, (const uint8_t*)nullptr, (const int*)W.large,
                       (const uint8_t*)W.cell_large);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_density_sign_backward(int64_t n_gauss, int64_t nv, const int* valid, const int64_t* prefix, const int* list,
                                 const float* samples, const float* pos, const float* rot, const float* scale,
                                 const float* opacity, const float* sh, DensityFilter flt, const int8_t* signs,
                                 float w, float* ws, hipStream_t st, const uint8_t* skip) {
    if (nv <= 0 || n_gauss <= 0) return 0;
    const DensityWs W(ws, n_gauss);
    hipLaunchKernelGGL(density_rows_kernel, dim3(nblk(n_gauss, 256)), dim3(256), 0, st, n_gauss, pos, rot, scale,
                       opacity, sh, flt, W.rows, W.large);
    if (std::fabs(w) >= SPLIT_MOST) hipLaunchKernelGGL(set_word_kernel, dim3(1), dim3(64), 0, st, W.large);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nv), dim3(256), 0, st, nv, valid, prefix, list, samples,
                           (const float4*)W.rows, sh, flt, signs, w, W.acc, skip, (const int*)W.large);
    };
    if (flt.ada) launch(density_sign_backward_kernel<true>);
    else launch(density_sign_backward_kernel<false>);
    hipLaunchKernelGGL(density_plain_backward_kernel<true>, dim3(std::min(nblk(nv, 64), 4096u)), dim3(64), 0, st, nv,
                       valid, prefix, list, samples, (const float4*)W.rows, sh, flt, (const float*)nullptr,
                       (const float*)nullptr, signs, w, (float*)nullptr, W.acc, skip, (const int*)W.large,
                       (const uint8_t*)nullptr);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_density_attr_grad(int64_t N, const float* rot, const float* scale, const float* gacc, DensityFilter flt,
                             float* dsh, float* dpos, float* drot, float* dscale, float* dopac, hipStream_t st) {
    if (N <= 0) return 0;
    hipLaunchKernelGGL(density_attr_grad_kernel, dim3(nblk(N, 256)), dim3(256), 0, st, N, rot, scale, gacc, flt, dsh, dpos,
                       drot, dscale, dopac);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_six_point_backward(int64_t N, int K, const NodeXf* table, const uint32_t* ends_idx, const float* ends_w,
                              const float* ends, const float* rot0, const float* scale0, const float* sh0,
                              const float* rot1, const float* scale1, const float* gr, const float* gacc,
                              DensityFilter flt, float pad, float coeff, const ShRotTables* Tsh, float* gends, float* drot0,
                              float* dscale0, hipStream_t st) {
    if (N <= 0) return 0;
    hipLaunchKernelGGL(six_point_backward_kernel, dim3(nblk(N, 128)), dim3(128), 0, st, N, K, table, ends_idx,
                       ends_w, ends, rot0, scale0, sh0, rot1, scale1, gr, gacc, flt, pad, coeff, Tsh, gends, drot0,
                       dscale0);
    HIP_RET(hipGetLastError());
    return 0;
}

size_t inverse_index_words(int64_t n_entries) {
    return (size_t)n_entries * 6 + radix_workspace_words(n_entries) + 64;
}

int build_inverse_index(int64_t n_end_entries, int64_t n_entries, int M, const uint32_t* ends_idx,
                        const uint32_t* sample_idx, uint32_t* ws, uint32_t* entries, uint2* rng, hipStream_t st) {
    if (n_entries <= 0 || n_entries > 0xffffffffll) return -1;
    uint64_t* keys = reinterpret_cast<uint64_t*>(ws);
    uint64_t* keys_alt = keys + n_entries;
    uint32_t* vals_alt = reinterpret_cast<uint32_t*>(keys_alt + n_entries);
    uint32_t* sort_ws = vals_alt + n_entries;
    hipLaunchKernelGGL(entry_keys_kernel, dim3(nblk(n_entries, 256)), dim3(256), 0, st, n_end_entries, n_entries,
                       ends_idx, sample_idx, keys, entries);
    HIP_RET(hipGetLastError());
    int bits = 1;
    while ((1ll << bits) < M) bits++;
    int rc = launch_radix_sort(keys, entries, keys_alt, vals_alt, n_entries, bits, sort_ws, st);
    if (rc) return rc;
    hipLaunchKernelGGL(zero_u32_kernel, dim3(nblk(2 * (int64_t)M, 256)), dim3(256), 0, st, (uint32_t*)rng,
                       2 * (int64_t)M);
    hipLaunchKernelGGL(node_ranges_kernel, dim3(nblk(n_entries, 256)), dim3(256), 0, st, keys, n_entries, M, rng);
    HIP_RET(hipGetLastError());
    return 0;
}

int launch_node_gather(int M, int K, int64_t n_end_entries, const uint2* rng, const uint32_t* entries,
                       const NodeXf* table, const float* ends_w, const float* ends0, const float* gends,
                       const float* sample_w, const float* samples0, const float* gsamp, NodeXf* dtable,
                       hipStream_t st) {
    if (M <= 0) return 0;
    hipLaunchKernelGGL(node_gather_kernel, dim3((unsigned)M), dim3(256), 0, st, M, K, n_end_entries, rng, entries,
                       table, ends_w, ends0, gends, sample_w, samples0, gsamp, dtable);
    HIP_RET(hipGetLastError());
    return 0;
}

}  // namespace arapgs
