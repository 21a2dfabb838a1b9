// Graph build on gfx950: farthest-point node sampling and the point -> node
// K-nearest search with the reference's exact tie semantics.
//
// The reference KNN (DeformGraph::findNearestNodes, Deform.hpp:153-185) is a
// selection sort over the first k slots of a position array: at step i it keeps
// slot i unless a strictly smaller distance exists, otherwise takes the
// highest-position minimum of the descending scan, then swaps slot i with the
// winner. This file reproduces the resulting index sequence bit for bit:
//   1. one pass over the nodes near the query (or, few nodes, all of them; they
//      are staged in LDS) keeps the smallest squared distances per query (exact
//      float arithmetic, no contraction);
//   2. if every node outside that list has a strictly larger sqrt-distance than
//      the k-th selected one, the selection sort is replayed on the candidates
//      only (positions start at the node index; non-candidates never win);
//   3. otherwise the query is flagged and a wave-cooperative kernel replays the
//      full selection sort over all M positions.
#pragma clang fp contract(off)
#include "common.hpp"
#include "grid.hpp"
#include "sort.hpp"

#include <algorithm>
#include <climits>
#include <mutex>
#include <numeric>

namespace arapgs {

namespace {

constexpr uint32_t KNN_DONE = 0xffffffffu;  // a flagged query that needs no replay any more
constexpr int L_TOP = 16;   // candidate list length (>= KNN_MAX + 1 + slack)
// Whether the search is by cells: what it costs grows with K, what visiting all
// nodes costs with their number; the sorting of a workgroup's nodes (about 10 us)
// is shared by more queries where there are many. All nodes and by cells, K = 8,
// 600k queries: 96 nodes 263 and 306 us, 160 nodes 358 and 328, 320 nodes 597 and
// 321; 1,000 queries: 160 nodes 114 and 139, 224 nodes 145 and 134. K = 1, 64
// nodes: 137 and 104, 53 and 52; K = 12, 256 nodes: 514 and 545, 166 and 213.
inline bool knn_by_cells(int M, int k, int64_t Q) {
    return M >= (Q > 300000 ? 40 + 7 * k * k / 4 : 60 + k * (k + 7));
}

// Exact distance of Deform.hpp:164-165: float differences, products summed left
// to right without contraction (this file is compiled with contraction off; the
// header intrinsics __fmul_rn/__fadd_rn are plain contractible ops here, so the
// expression is written out), correctly rounded sqrt.
__device__ __forceinline__ float knn_d2(float px, float py, float pz, float nx, float ny, float nz) {
    const float a = px - nx, b = py - ny, c = pz - nz;
    return (a * a + b * b) + c * c;
}

// Weights of DeformGraph::computeWeights (Deform.hpp:187-208) in double from the
// float distances of the selected slots; written as float.
__device__ __forceinline__ void write_weights(const float* dsel, int k, float* w) {
    const double dmax = (double)dsel[k];
    double wd[KNN_MAX_T];
    double sum = 0.0;
    for (int j = 0; j < k; j++) {
        const double x = 1.0 - (double)dsel[j] / dmax;
        wd[j] = x * x;
        sum += wd[j];
    }
    if (k == 1) { w[0] = 1.0f; return; }
    for (int j = 0; j < k; j++) w[j] = (float)(wd[j] / sum);
}

// Step 2 for query q with its L smallest squared distances td, ascending, and their
// nodes ti (-1: fewer); `all`: no node was left out of them. False: step 3 is needed.
template <int K, int L>
__device__ __forceinline__ bool knn_select(int64_t q, const float (&td)[L], const int (&ti)[L], bool all,
                                           uint32_t* __restrict__ out_idx, float* __restrict__ out_w) {
    constexpr int KK = K + 1;  // slots selected by the reference (k_nearest + 1)
    // sqrt distances of the kept candidates: ascending d2, so non-decreasing
    float sd[L];
#pragma unroll
    for (int s = 0; s < L; s++) sd[s] = ti[s] >= 0 ? __builtin_sqrtf(td[s]) : __builtin_inff();
    const float T = sd[KK - 1];
    const bool complete = all || (sd[L - 1] > T);
    if (!complete) return false;
    // Replay the selection sort on the candidates (value <= T); every node not
    // kept has a larger value, so it can neither win nor tie.
    int pos[L];
    bool alive[L];
#pragma unroll
    for (int s = 0; s < L; s++) { pos[s] = ti[s]; alive[s] = (ti[s] >= 0) && (sd[s] <= T); }
    float dsel[KK];
    uint32_t* oq = out_idx + q * KK;
#pragma unroll
    for (int i = 0; i < KK; i++) {
        float mv = __builtin_inff();
#pragma unroll
        for (int s = 0; s < L; s++)
            if (alive[s] && sd[s] < mv) mv = sd[s];
        int at_i = -1, win = -1, best_pos = -1;
#pragma unroll
        for (int s = 0; s < L; s++) {
            if (!alive[s]) continue;
            if (pos[s] == i) at_i = s;
            if (sd[s] == mv && pos[s] > best_pos) { best_pos = pos[s]; win = s; }
        }
        // slot i keeps its element unless something is strictly smaller
        if (at_i >= 0 && sd[at_i] == mv) win = at_i;
        int wpos = 0, wid = 0;
        float wv = 0.0f;
#pragma unroll
        for (int s = 0; s < L; s++)
            if (s == win) { wpos = pos[s]; wid = ti[s]; wv = sd[s]; }
        oq[i] = (uint32_t)wid;
        dsel[i] = wv;
#pragma unroll
        for (int s = 0; s < L; s++) {
            if (s == win) { pos[s] = i; alive[s] = false; }
            else if (s == at_i) pos[s] = wpos;  // element at slot i moves to the winner's slot
        }
    }
    if (out_w) {
        const double dmax = (double)dsel[K];
        double wd[K];
        double sum = 0.0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const double x = 1.0 - (double)dsel[j] / dmax;
            wd[j] = x * x;
            sum += wd[j];
        }
        float* wq = out_w + q * K;
        if (K == 1) wq[0] = 1.0f;
        else {
#pragma unroll
            for (int j = 0; j < K; j++) wq[j] = (float)(wd[j] / sum);
        }
    }
    return true;
}

// A query for step 3.
__device__ __forceinline__ void knn_flag(int64_t q, uint32_t* __restrict__ fallback_list,
                                         uint32_t* __restrict__ fallback_count) {
    fallback_list[atomicAdd(fallback_count, 1u)] = (uint32_t)q;
}

// The L nearest nodes found so far, ascending.
template <int L>
struct KnnList {
    float d[L];
    int id[L];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int s = 0; s < L; s++) { d[s] = __builtin_inff(); id[s] = -1; }
    }
    __device__ __forceinline__ void add(float v, int node) {
        if (!(v < d[L - 1])) return;
#pragma unroll
        for (int s = 0; s < L; s++) {
            if (v < d[s]) {
                const float tv = d[s]; d[s] = v; v = tv;
                const int ti = id[s]; id[s] = node; node = ti;
            }
        }
    }
};

template <int K>
__global__ void __launch_bounds__(256) knn_main_kernel(const float* __restrict__ nodes, int M,
                                                       const float* __restrict__ queries, int64_t Q,
                                                       uint32_t* __restrict__ out_idx, float* __restrict__ out_w,
                                                       uint32_t* __restrict__ fallback_list,
                                                       uint32_t* __restrict__ fallback_count) {
    extern __shared__ float s_nodes[];  // 3*M
    for (int i = threadIdx.x; i < 3 * M; i += blockDim.x) s_nodes[i] = nodes[i];
    __syncthreads();
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= Q) return;
    const float px = queries[3 * q], py = queries[3 * q + 1], pz = queries[3 * q + 2];
    KnnList<L_TOP> near;
    near.clear();
    for (int j = 0; j < M; j++)
        near.add(knn_d2(px, py, pz, s_nodes[3 * j], s_nodes[3 * j + 1], s_nodes[3 * j + 2]), j);
    if (!knn_select<K>(q, near.d, near.id, M <= L_TOP, out_idx, out_w)) knn_flag(q, fallback_list, fallback_count);
}

// The same search over the nodes near each query only. Every workgroup sorts the
// nodes into a uniform grid of about M cells over their bounding box in LDS
// (KNN_CELLS_MAX starts and 16 bytes a node: no scratch memory, so it also serves
// arapgs_knn_noalloc). A thread searches the 27 cells around its query (more,
// while they hold no K + 1 nodes), and then those of the box that holds every
// node as near as the (K + 1)-th found: the result is that of the search over all
// nodes, whatever the order of the visits. Rows of cells along z are contiguous.
// Where the box is estimated at more than half of all nodes (a row of cells is
// taken for KNN_ROW nodes, and 80 for the list's second start), and for queries
// away from the nodes by half of their box's longest side, all nodes are visited,
// in steps of a fraction of M: in cell order they would tend to come ever nearer,
// and each enter the list. 200k queries, 2048 nodes in a cube, a plane and a line
// of the same length, K = 8, all nodes for every query | growing blocks of cells
// alone | this: 0.3 of half a side away 5.0 | 0.75 | 0.42 ms, 4.9 | 15.6 | 1.3 ms,
// 4.6 | 276 | 1.3 ms. 6M queries among 2048 nodes: 44 ms with all nodes for every
// query, 3.3 ms (95% of the vector issue: FP32 distances and the list).
constexpr int KNN_CELLS_MAX = 4096;
constexpr int KNN_SHELLS = 3;
constexpr int KNN_ROW = 2;

struct KnnCells {
    const float4* pts;      // (x, y, z, node) in cell order
    const uint32_t* ends;   // of the cells
    float mn[3], edge, slack;
    int n[3], M, step;

    __device__ __forceinline__ int cell(float p, int c) const {
        return (int)fminf(fmaxf(floorf((p - mn[c]) / edge), 0.0f), (float)(n[c] - 1));
    }
    // The nearest nodes of p, of which every one as near as the (K + 1)-th is there or the list is full.
    // Passes over boxes of cells, each without the box before it; one place in the code adds to the list
    // (its registers would be held once for each).
    template <int K, int L>
    __device__ __forceinline__ void search(const float (&p)[3], KnnList<L>& near) const {
        const int c[3] = {cell(p[0], 0), cell(p[1], 1), cell(p[2], 2)};
        near.clear();
        int lo[3], hi[3], had_lo[3], had_hi[3];  // the box, and the part of it that has been visited
        float out2[3];                           // squared distances to the nodes' box, less the slack
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = max(c[k] - 1, 0);
            hi[k] = min(c[k] + 1, n[k] - 1);
            had_lo[k] = 0;
            had_hi[k] = -1;
            const float o = fmaxf(fmaxf(mn[k] - p[k], p[k] - (mn[k] + (float)n[k] * edge)) - slack, 0.0f);
            out2[k] = o * o;
        }
        const float half = 0.5f * (float)max(n[0], max(n[1], n[2])) * edge;
        bool all = out2[0] + out2[1] + out2[2] > half * half, last = all;
        if (all) lo[0] = hi[0] = lo[1] = hi[1] = 0;
        for (int r = 1;; r++) {
            for (int x = lo[0]; x <= hi[0]; x++)
                for (int y = lo[1]; y <= hi[1]; y++) {
                    const int row = (x * n[1] + y) * n[2];
                    const bool had = x >= had_lo[0] && x <= had_hi[0] && y >= had_lo[1] && y <= had_hi[1];
                    for (int side = 0; side < (had ? 2 : 1); side++) {
                        const int z0 = side ? had_hi[2] + 1 : lo[2], z1 = had && !side ? had_lo[2] - 1 : hi[2];
                        int j = row + z0 > 0 && z0 <= z1 ? (int)ends[row + z0 - 1] : 0;
                        int count = z0 <= z1 ? (int)ends[row + z1] - j : 0;
                        if (all) { j = 0; count = M; }
                        const int inc = all ? step : 1;
                        for (; count > 0; count--) {
                            const float4 v = pts[j];
                            near.add(knn_d2(p[0], p[1], p[2], v.x, v.y, v.z), __float_as_int(v.w));
                            j += inc;
                            if (j >= M) j -= M;
                        }
                    }
                }
            if (last) return;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                had_lo[k] = lo[k];
                had_hi[k] = hi[k];
            }
            bool held = true;  // the next box was visited
            if (r < KNN_SHELLS && !(near.d[K] < __builtin_inff())) {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    lo[k] = max(c[k] - r - 1, 0);
                    hi[k] = min(c[k] + r + 1, n[k] - 1);
                    held = held && lo[k] == had_lo[k] && hi[k] == had_hi[k];
                }
            } else {
                last = true;
                // in a direction, less what the query is away from the nodes' box in the others; the margin
                // keeps every node outside strictly farther after the square root too
                const float most = near.d[K] * 1.00001f;
                int seen = 1;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const float left = most - (out2[0] + out2[1] + out2[2] - out2[k]);
                    const float reach = left >= 0.0f ? __builtin_sqrtf(left) + slack : __builtin_inff();
                    lo[k] = cell(p[k] - reach, k);
                    hi[k] = cell(p[k] + reach, k);
                    held = held && lo[k] >= had_lo[k] && hi[k] <= had_hi[k];
                    seen *= min(hi[k], had_hi[k]) - max(lo[k], had_lo[k]) + 1;
                }
                const int rows = (hi[0] - lo[0] + 1) * (hi[1] - lo[1] + 1);
                if (!held &&
                    (rows * (hi[2] - lo[2] + 1) - seen) * M > (M / 2 + 80 - KNN_ROW * rows) * (n[0] * n[1] * n[2])) {
                    all = true;
                    near.clear();
                    lo[0] = hi[0] = lo[1] = hi[1] = 0;
                    had_hi[0] = -1;
                }
            }
            if (held) return;
        }
    }
};

// L: K + 4 entries are enough but where many nodes lie at the K-th distance (nodes
// on a lattice), and keep more queries in flight. The queries flagged for that
// are searched AGAIN with L_TOP of them, in a launch of its own, which without any
// ends at once: in one kernel the longer list's registers cost every query a third
// (600k queries, 256 nodes, K = 8: 0.34 -> 0.47 ms). 200k queries at the face
// centres of a lattice of 1728 nodes, K = 8: 49 ms replayed one by one, 0.25 ms so
// (4.2 ms with the longer list over all nodes).
template <int K, int L, bool AGAIN>
__global__ void __launch_bounds__(256) knn_cells_kernel(const float* __restrict__ nodes, int M,
                                                        const float* __restrict__ queries, int64_t Q,
                                                        uint32_t* __restrict__ out_idx, float* __restrict__ out_w,
                                                        uint32_t* __restrict__ fallback_list,
                                                        uint32_t* __restrict__ fallback_count, int step) {
    extern __shared__ float4 s_pts[];  // M nodes (x, y, z, id) in cell order, then the cells' starts
    __shared__ float s_red[6][4];
    __shared__ float s_geom[5];        // box minimum, cell edge, slack of the bounds
    __shared__ int s_dim[4], s_scan[4];
    uint32_t* s_start = reinterpret_cast<uint32_t*>(s_pts + M);
    if (AGAIN) {
        Q = *fallback_count;
        if ((int64_t)blockIdx.x * 256 >= Q) return;
    }
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()}, hi[3] = {-lo[0], -lo[0], -lo[0]};
    for (int i = t; i < M; i += 256)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            lo[c] = fminf(lo[c], nodes[3 * i + c]);
            hi[c] = fmaxf(hi[c], nodes[3 * i + c]);
        }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[c] = fminf(lo[c], __shfl_xor(lo[c], o));
            hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o));
        }
        if (lane == 0) {
            s_red[c][wave] = lo[c];
            s_red[3 + c][wave] = hi[c];
        }
    }
    __syncthreads();
    if (t == 0) {
        float ext[3], big = 0.0f, far = 0.0f;
        for (int c = 0; c < 3; c++) {
            const float a = fminf(fminf(s_red[c][0], s_red[c][1]), fminf(s_red[c][2], s_red[c][3]));
            const float b = fmaxf(fmaxf(s_red[3 + c][0], s_red[3 + c][1]), fmaxf(s_red[3 + c][2], s_red[3 + c][3]));
            s_geom[c] = a;
            ext[c] = b - a;
            big = fmaxf(big, ext[c]);
            far = fmaxf(far, fmaxf(fabsf(a), fabsf(b)));
        }
        const float v = fmaxf(ext[0], 1e-3f * big) * fmaxf(ext[1], 1e-3f * big) * fmaxf(ext[2], 1e-3f * big);
        float edge = cbrtf(v / (float)M);
        // a box without a finite size, and one that rounding would blur, is one cell
        const bool one = !(edge > 1e-5f * far) || !(edge < 3e38f);
        int dim[3] = {1, 1, 1};
        while (!one) {
            bool fits = true;
            for (int c = 0; c < 3; c++) {
                const float d = floorf(ext[c] / edge) + 1.0f;
                fits = fits && d <= (float)KNN_CELLS_MAX;
                dim[c] = fits ? (int)d : 1;
            }
            if (fits && (int64_t)dim[0] * dim[1] * dim[2] <= KNN_CELLS_MAX) break;
            edge *= 1.1f;
        }
        for (int c = 0; c < 3; c++) s_dim[c] = dim[c];
        s_dim[3] = dim[0] * dim[1] * dim[2];
        s_geom[3] = edge;
        // a node may lie this far outside its cell (rounding of its coordinates)
        s_geom[4] = 1e-2f * edge + 1e-6f * far;
    }
    __syncthreads();
    const float mn0 = s_geom[0], mn1 = s_geom[1], mn2 = s_geom[2], edge = s_geom[3], slack = s_geom[4];
    const int n0 = s_dim[0], n1 = s_dim[1], n2 = s_dim[2], nc = s_dim[3];
    const auto cell = [&](float p, float mn, int n) { return (int)fminf(fmaxf(floorf((p - mn) / edge), 0.0f), (float)(n - 1)); };
    for (int i = t; i <= nc; i += 256) s_start[i] = 0u;
    __syncthreads();
    for (int i = t; i < M; i += 256)
        atomicAdd(&s_start[(cell(nodes[3 * i], mn0, n0) * n1 + cell(nodes[3 * i + 1], mn1, n1)) * n2 +
                           cell(nodes[3 * i + 2], mn2, n2)], 1u);
    __syncthreads();
    {
        // each thread's run of cells, the threads' sums scanned; the starts end
        // one run further (the scatter below moves each to its cell's end)
        const int per = (nc + 255) / 256, c0 = min(t * per, nc), c1 = min(c0 + per, nc);
        uint32_t sum = 0;
        for (int i = c0; i < c1; i++) sum += s_start[i];
        uint32_t x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63) s_scan[wave] = (int)x;
        __syncthreads();
        uint32_t run = x - sum;
        for (int w = 0; w < wave; w++) run += (uint32_t)s_scan[w];
        for (int i = c0; i < c1; i++) {
            const uint32_t n = s_start[i];
            s_start[i] = run;
            run += n;
        }
    }
    __syncthreads();
    for (int i = t; i < M; i += 256) {
        const float x = nodes[3 * i], y = nodes[3 * i + 1], z = nodes[3 * i + 2];
        const uint32_t at = atomicAdd(&s_start[(cell(x, mn0, n0) * n1 + cell(y, mn1, n1)) * n2 + cell(z, mn2, n2)], 1u);
        s_pts[at] = make_float4(x, y, z, __int_as_float(i));
    }
    __syncthreads();
    // s_start[c] is now the end of cell c: its nodes are [s_start[c - 1], s_start[c])
    const KnnCells C{s_pts, s_start, {mn0, mn1, mn2}, edge, slack, {n0, n1, n2}, M, step};
    for (int64_t i = (int64_t)blockIdx.x * 256 + t; i < Q; i += (int64_t)gridDim.x * 256) {
        const int64_t q = AGAIN ? fallback_list[i] : i;
        const float p[3] = {queries[3 * q], queries[3 * q + 1], queries[3 * q + 2]};
        KnnList<L> near;
        C.search<K>(p, near);
        const bool found = knn_select<K>(q, near.d, near.id, false, out_idx, out_w);
        if (AGAIN && found) fallback_list[i] = KNN_DONE;
        if (!AGAIN && !found) knn_flag(q, fallback_list, fallback_count);
    }
}

// Exact fallback: one wave per flagged query replays the full selection sort.
// Swapped positions are tracked in a small override table (<= 2(k+1) entries).
__global__ void __launch_bounds__(64) knn_fallback_kernel(const float* __restrict__ nodes, int M,
                                                          const float* __restrict__ queries, int k,
                                                          uint32_t* __restrict__ out_idx, float* __restrict__ out_w,
                                                          const uint32_t* __restrict__ fallback_list,
                                                          const uint32_t* __restrict__ fallback_count) {
    const uint32_t n_fb = *fallback_count;
    const int kk = k + 1;
    __shared__ int ov_pos[2 * (KNN_MAX_T + 1)], ov_el[2 * (KNN_MAX_T + 1)];
    __shared__ int n_ov;
    __shared__ float red_v[64];
    __shared__ int red_p[64];
    // every gridDim.x-th query, 64 of the list read at a time
    for (int64_t f0 = blockIdx.x; f0 < n_fb; f0 += 64 * (int64_t)gridDim.x) {
      const int64_t f = f0 + threadIdx.x * (int64_t)gridDim.x;
      const uint32_t mine = f < n_fb ? fallback_list[f] : KNN_DONE;
      for (uint64_t left = __ballot(mine != KNN_DONE); left != 0ull; left &= left - 1ull) {
        const int64_t q = (uint32_t)__builtin_amdgcn_readlane((int)mine, __builtin_ctzll(left));
        const float px = queries[3 * q], py = queries[3 * q + 1], pz = queries[3 * q + 2];
        if (threadIdx.x == 0) n_ov = 0;
        __syncthreads();
        float dsel[KNN_MAX_T + 1];
        for (int i = 0; i < kk; i++) {
            // element currently at position p
            auto elem_at = [&](int p) {
                int e = p;
                for (int o = 0; o < n_ov; o++)
                    if (ov_pos[o] == p) e = ov_el[o];
                return e;
            };
            float bv = __builtin_inff();
            int bp = -1;  // priority: position i beats all, then higher positions
            for (int p = i + (int)threadIdx.x; p < M; p += 64) {
                const int e = elem_at(p);
                const float v = __builtin_sqrtf(knn_d2(px, py, pz, nodes[3 * e], nodes[3 * e + 1], nodes[3 * e + 2]));
                const int pr = (p == i) ? 0x7fffffff : p;
                if (v < bv || (v == bv && pr > bp)) { bv = v; bp = pr; }
            }
            red_v[threadIdx.x] = bv;
            red_p[threadIdx.x] = bp;
            __syncthreads();
            if (threadIdx.x == 0) {
                float v = red_v[0];
                int pr = red_p[0];
                for (int l = 1; l < 64; l++)
                    if (red_v[l] < v || (red_v[l] == v && red_p[l] > pr)) { v = red_v[l]; pr = red_p[l]; }
                const int wpos = (pr == 0x7fffffff) ? i : pr;
                const int we = elem_at(wpos), ie = elem_at(i);
                out_idx[q * kk + i] = (uint32_t)we;
                red_v[0] = v;
                // swap elements at positions i and wpos
                int have_i = -1, have_w = -1;
                for (int o = 0; o < n_ov; o++) {
                    if (ov_pos[o] == i) have_i = o;
                    if (ov_pos[o] == wpos) have_w = o;
                }
                if (have_i < 0) { have_i = n_ov; ov_pos[n_ov++] = i; }
                ov_el[have_i] = we;
                if (wpos != i) {
                    if (have_w < 0) { have_w = n_ov; ov_pos[n_ov++] = wpos; }
                    ov_el[have_w] = ie;
                }
            }
            __syncthreads();
            dsel[i] = red_v[0];
            __syncthreads();
        }
        if (out_w && threadIdx.x == 0) write_weights(dsel, k, out_w + q * k);
        __syncthreads();
      }
    }
}

// ---------------------------------------------------------------- FPS
// farthest_control_points_sampling (helper.cpp:139-177): distances as
// pts_distance (helper.cpp:60-63) — float differences, squares summed in double,
// double sqrt rounded to float; running min with strict '<'; argmax keeps the
// first maximum (std::max_element).

// FetchFirstNodeIdx (helper.cpp:180-195): argmax of x+y+z (float, first max,
// initial -100000).
__global__ void fps_first_kernel(const float* __restrict__ pos, int64_t N, unsigned long long* __restrict__ best) {
    // packed key: larger sum first, then smaller index
    __shared__ unsigned long long red[256];
    unsigned long long local = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        const float s = (0.0f + pos[3 * i]) + pos[3 * i + 1] + pos[3 * i + 2];
        if (!(s > -100000.0f)) continue;
        uint32_t b = __float_as_uint(s);
        b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);  // order-preserving map
        const unsigned long long key = ((unsigned long long)b << 32) | (uint32_t)(0xffffffffu - (uint32_t)i);
        local = local > key ? local : key;
    }
    red[threadIdx.x] = local;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] > red[threadIdx.x + s] ? red[threadIdx.x] : red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicMax(best, red[0]);
}

__global__ void fps_clear_kernel(unsigned long long* __restrict__ best) {
    if (threadIdx.x == 0) *best = 0ull;
}

// Points in spatial order: the cell of a 1024^3 grid over
// [lo, hi] as an interleaved (Morton) key of 30 bits.
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    return (v | (v << 2)) & 0x09249249u;
}

__global__ void fps_keys_kernel(const float* __restrict__ pos, int64_t N, const float* __restrict__ box,
                                uint32_t* __restrict__ keys, uint32_t* __restrict__ ids) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float ext = fmaxf(fmaxf(box[3] - box[0], box[4] - box[1]), box[5] - box[2]);
    uint32_t k = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const float u = (pos[3 * i + c] - box[c]) / ext * 1024.0f;
        k |= spread10((uint32_t)fminf(fmaxf(u, 0.0f), 1023.0f)) << c;
    }
    keys[i] = k;
    ids[i] = (uint32_t)i;
}

// out[0], the points with their running minimum distance (x, y, z, d) for the
// full steps (pts, may be null) and cleared words.
__global__ void fps_init_kernel(const float* __restrict__ pos, int64_t N, float4* __restrict__ pts,
                                unsigned long long* __restrict__ zero, int64_t n_zero,
                                const unsigned long long* __restrict__ best, int* __restrict__ out,
                                unsigned int* __restrict__ counter) {
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    if (pts)
        for (int64_t i = i0; i < N; i += stride)
            pts[i] = make_float4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], 3.402823466e+38f);
    for (int64_t i = i0; i < n_zero; i += stride) zero[i] = 0ull;
    if (i0 == 0) {
        const unsigned long long b = *best;
        out[0] = b == 0 ? 0 : (int)(0xffffffffu - (uint32_t)(b & 0xffffffffu));
        *counter = 0;
    }
}

// Folds the chosen point l into a point's running minimum d: float differences,
// squares summed in double, double root rounded to float, strict '<'. The root
// is skipped where the sum is clearly larger. True if d changed.
__device__ __forceinline__ bool fps_fold(float px, float py, float pz, float& d, float lx, float ly, float lz) {
    const float dx = lx - px, dy = ly - py, dz = lz - pz;
    const double s = ((double)dx * (double)dx + (double)dy * (double)dy) + (double)dz * (double)dz;
    const double w = (double)d;
    if (s > w * w * 1.000001) return false;
    const float r = (float)__builtin_sqrt(s);
    if (!(r < d)) return false;
    d = r;
    return true;
}

// distances are >= 0: float bits order like unsigned ints; the first index wins ties
__device__ __forceinline__ unsigned long long fps_key(float d, uint32_t id) {
    return ((unsigned long long)__float_as_uint(d) << 32) | (0xffffffffu - id);
}

// A key of the one-launch form as a word with the number of its step: 31 bits of
// distance, 22 of index, 11 of the step counted from 1.
constexpr int FPS_ID_BITS = 22, FPS_TAG_BITS = 11;
__device__ __forceinline__ unsigned long long fps_word(unsigned long long key, int step) {
    const uint32_t id = 0xffffffffu - (uint32_t)key;
    return (key >> 32) << (FPS_ID_BITS + FPS_TAG_BITS) |
           (unsigned long long)(((1u << FPS_ID_BITS) - 1u) - id) << FPS_TAG_BITS |
           ((uint32_t)(step + 1) & ((1u << FPS_TAG_BITS) - 1u));
}
__device__ __forceinline__ int fps_word_id(unsigned long long word) {
    constexpr uint32_t mask = (1u << FPS_ID_BITS) - 1u;
    return (int)(mask - ((uint32_t)(word >> FPS_TAG_BITS) & mask));
}

// Wave maxima by DPP (row shifts, then the rows' last lanes broadcast): a dozen
// vector instructions instead of twelve trips through the LDS pipe.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#define ARAPGS_DPP_MAX(ctrl) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xf, 0xf, false))
    ARAPGS_DPP_MAX(0x111);  // row_shr:1
    ARAPGS_DPP_MAX(0x112);  // row_shr:2
    ARAPGS_DPP_MAX(0x114);  // row_shr:4
    ARAPGS_DPP_MAX(0x118);  // row_shr:8
    ARAPGS_DPP_MAX(0x142);  // row_bcast:15
    ARAPGS_DPP_MAX(0x143);  // row_bcast:31
#undef ARAPGS_DPP_MAX
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ unsigned long long wave_max64(unsigned long long v) {
    const uint32_t hi = wave_max_u32((uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | wave_max_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : 0u);
}

// One FPS step over all points: fold the last chosen point into the running
// minima and find the first maximum; the last block to finish writes out[step+1]
// (one block per CU: the blocks' arrivals at the counter take turns).
__global__ void __launch_bounds__(1024) fps_step_kernel(const float* __restrict__ pos, int64_t N,
                                                        float4* __restrict__ pts, int step, int* __restrict__ out,
                                                       unsigned long long* __restrict__ partial,
                                                       unsigned int* __restrict__ counter) {
    const int last = out[step];
    const float lx = pos[3 * (int64_t)last], ly = pos[3 * (int64_t)last + 1], lz = pos[3 * (int64_t)last + 2];
    unsigned long long local = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        float4 p = pts[i];
        if (fps_fold(p.x, p.y, p.z, p.w, lx, ly, lz)) pts[i].w = p.w;
        const unsigned long long key = fps_key(p.w, (uint32_t)i);
        local = local > key ? local : key;
    }
    __shared__ unsigned long long red[16];
    __shared__ bool is_last;
    local = wave_max64(local);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) local = local > red[w] ? local : red[w];
        partial[blockIdx.x] = local;
        __threadfence();
        const unsigned int done = atomicAdd(counter, 1u);
        is_last = (done == gridDim.x - 1);
    }
    __syncthreads();
    if (is_last) {
        __threadfence();
        unsigned long long v = 0;
        for (unsigned int b = threadIdx.x; b < gridDim.x; b += blockDim.x) {
            const unsigned long long p = __hip_atomic_load(&partial[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v = v > p ? v : p;
        }
        v = wave_max64(v);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < 16; w++) v = v > red[w] ? v : red[w];
            out[step + 1] = (int)(0xffffffffu - (uint32_t)(v & 0xffffffffu));
            *counter = 0;
        }
    }
}

// All steps in one launch. The points, in spatial order, live in registers (12 a
// thread, 768 consecutive ones a wave); a chosen point lowers the minima only
// near itself, so a wave whose bounding sphere is not nearer to it than the
// wave's largest minimum skips the step (its minima would all stay, whatever the
// point: the choices are those of the full steps bit for bit). Per step every
// workgroup publishes its maximum (distance and index, and the three
// coordinates: four words that carry the step's number) and reads all the
// others': one trip through memory, no grid barrier, no cache write-back, no
// launch. Two sets of words take turns: a workgroup publishes step s + 2 after it
// has read every word of step s + 1, whose writers had read all of step s by
// then. The wait is bounded: a workgroup
// that misses another's words for `polls` polls (the workgroups could not all
// run at once) ends the kernel with *failed set, and the caller takes the steps
// one launch each.
constexpr int FPS_PT = 12, FPS_WG = 1024 * FPS_PT, FPS_MAX_WGS = 256;
static_assert((int64_t)FPS_WG * FPS_MAX_WGS < 1 << FPS_ID_BITS, "point indices of the one-launch form");

__global__ void __launch_bounds__(1024) fps_resident_kernel(const float* __restrict__ pos, int64_t N,
                                                            const uint32_t* __restrict__ ids, int steps,
                                                            int* __restrict__ out,
                                                            unsigned long long* __restrict__ slots, int polls,
                                                            int* __restrict__ failed) {
    __shared__ unsigned long long s_word[4 * FPS_MAX_WGS];
    __shared__ unsigned long long s_key[16];
    __shared__ float s_pos[16][3];
    __shared__ int s_fail;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, W = gridDim.x;
    const int64_t base = (int64_t)blockIdx.x * FPS_WG + wave * (64 * FPS_PT) + lane;
    float x[FPS_PT], y[FPS_PT], z[FPS_PT], d[FPS_PT];
    uint32_t id[FPS_PT];
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()}, hi[3] = {-lo[0], -lo[0], -lo[0]};
#pragma unroll
    for (int j = 0; j < FPS_PT; j++) {
        const int64_t i = base + 64 * j;
        const bool in = i < N;
        id[j] = in ? ids[i] : 0xffffffffu;  // key 0: never chosen
        const int64_t g = in ? id[j] : ids[N - 1];
        x[j] = pos[3 * g]; y[j] = pos[3 * g + 1]; z[j] = pos[3 * g + 2];
        d[j] = in ? 3.402823466e+38f : 0.0f;
        lo[0] = fminf(lo[0], x[j]); lo[1] = fminf(lo[1], y[j]); lo[2] = fminf(lo[2], z[j]);
        hi[0] = fmaxf(hi[0], x[j]); hi[1] = fmaxf(hi[1], y[j]); hi[2] = fmaxf(hi[2], z[j]);
    }
    float c[3], r2 = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], o));
        }
        c[k] = 0.5f * (lo[k] + hi[k]);
    }
    bool odd = false;  // a point without finite coordinates: the wave takes every step
#pragma unroll
    for (int j = 0; j < FPS_PT; j++) {
        const float dx = x[j] - c[0], dy = y[j] - c[1], dz = z[j] - c[2];
        const float s = dx * dx + dy * dy + dz * dz;
        odd = odd || !(s < 1e37f);
        r2 = fmaxf(r2, s);
    }
    for (int o = 32; o > 0; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
    const float radius = __ballot(odd) ? __builtin_nanf("") : __builtin_sqrtf(r2) * 1.00001f;
    float most = 3.402823466e+38f;  // the wave's largest minimum
    int64_t last = out[0];
    float lx = pos[3 * last], ly = pos[3 * last + 1], lz = pos[3 * last + 2];
    if (t == 0) s_fail = 0;
    __syncthreads();
    for (int step = 0; step < steps; step++) {
        // every point of the wave is at least |l - c| - radius away; the margin covers rounding
        const float ex = lx - c[0], ey = ly - c[1], ez = lz - c[2];
        const float dist = __builtin_sqrtf(ex * ex + ey * ey + ez * ez);
        if (step == 0 || !((dist - radius) * 0.99999f - 1e-6f * dist >= most)) {
            unsigned long long key = 0;
            float bx = 0.0f, by = 0.0f, bz = 0.0f;
#pragma unroll
            for (int j = 0; j < FPS_PT; j++) {
                fps_fold(x[j], y[j], z[j], d[j], lx, ly, lz);
                const unsigned long long k = id[j] == 0xffffffffu ? 0ull : fps_key(d[j], id[j]);
                if (k > key) {
                    key = k;
                    bx = x[j]; by = y[j]; bz = z[j];
                }
            }
            const unsigned long long best = wave_max64(key);
            most = __uint_as_float((uint32_t)(best >> 32));
            if (best == 0ull) {
                if (lane == 0) s_key[wave] = 0ull;  // a wave past the last point
            } else if (key == best) {               // one lane: indices differ
                s_key[wave] = best;
                s_pos[wave][0] = bx; s_pos[wave][1] = by; s_pos[wave][2] = bz;
            }
        }
        __syncthreads();
        // the workgroup's maximum: four words, written by four lanes
        if (wave == 0) {
            const unsigned long long k = lane < 16 ? s_key[lane] : 0ull;
            const unsigned long long best = wave_max64(k);
            const int w = best == 0ull ? 0 : (int)__builtin_ctzll(__ballot(k == best));
            if (lane < 4) {
                const unsigned long long word = lane == 0 ? fps_word(best, step)
                                                          : (unsigned long long)(step + 1) << 32 |
                                                                __float_as_uint(s_pos[w][lane - 1]);
                if (W == 1)
                    s_word[lane] = word;
                else
                    __hip_atomic_store(&slots[((step & 1) * W + blockIdx.x) * 4 + lane], word, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (W > 1 && t < 4 * W) {
            const unsigned long long* slot = &slots[(step & 1) * W * 4 + t];
            const int from = (t & 3) == 0 ? 0 : 32;  // where the step's number is, and how much of it
            const uint32_t mask = (t & 3) == 0 ? (1u << FPS_TAG_BITS) - 1u : 0xffffffffu;
            const uint32_t tag = (uint32_t)(step + 1) & mask;
            unsigned long long v = 0;
            bool there = false;
            for (int n = 0; !there && n < polls; n++) {
                v = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                there = ((uint32_t)(v >> from) & mask) == tag;
            }
            s_word[t] = v;
            if (!there) s_fail = 1;
        }
        __syncthreads();
        if (s_fail) {  // uniform: every wave of the workgroup leaves here
            if (t == 0) *failed = 1;
            return;
        }
        unsigned long long best = 0;
        int bw = 0;
        for (int w = lane; w < W; w += 64)
            if (s_word[4 * w] > best) {
                best = s_word[4 * w];
                bw = w;
            }
        const unsigned long long top = wave_max64(best);
        bw = __builtin_amdgcn_readlane(bw, (int)__builtin_ctzll(__ballot(best == top)));
        lx = __uint_as_float((uint32_t)s_word[4 * bw + 1]);
        ly = __uint_as_float((uint32_t)s_word[4 * bw + 2]);
        lz = __uint_as_float((uint32_t)s_word[4 * bw + 3]);
        if (blockIdx.x == 0 && t == 0) out[step + 1] = fps_word_id(top);
        // s_word is written again only after the next barrier, s_key and s_pos after this one's
    }
}

__global__ void clear_count_kernel(uint32_t* __restrict__ count) {
    if (threadIdx.x == 0) *count = 0u;
}

}  // namespace

// ---------------------------------------------------------------- launchers
int launch_knn(const float* nodes, int M, const float* queries, int64_t Q, int k, uint32_t* out_idx, float* out_w,
               uint32_t* scratch_list, uint32_t* scratch_count, hipStream_t st) {
    if (Q == 0) return 0;
    const size_t lds = sizeof(float) * 3 * (size_t)M;
    const size_t lds_cells = sizeof(float4) * (size_t)M + sizeof(uint32_t) * (KNN_CELLS_MAX + 1);
    const bool cells = knn_by_cells(M, k, Q);
    int step = (int)(0.618 * M);  // and no divisor in common with M: multiples of it mod M are all nodes
    while (std::gcd(step, M) != 1) step++;
    // a kernel, not a memset, clears the count: callers may capture the launches
    hipLaunchKernelGGL(clear_count_kernel, dim3(1), dim3(64), 0, st, scratch_count);
    const int64_t blocks = (Q + 255) / 256;
    switch (k) {
#define ARAPGS_KNN_CASE(KV)                                                                                         \
    case KV:                                                                                                        \
        if (cells) {                                                                                                \
            constexpr int L = KV <= 8 ? KV + 4 : L_TOP;                                                             \
            hipLaunchKernelGGL((knn_cells_kernel<KV, L, false>), dim3((unsigned)std::min<int64_t>(blocks, 1024)),   \
                               dim3(256), lds_cells, st, nodes, M, queries, Q, out_idx, out_w, scratch_list,        \
                               scratch_count, step);                                                                \
            if constexpr (L < L_TOP)                                                                                \
                hipLaunchKernelGGL((knn_cells_kernel<KV, L_TOP, true>), dim3((unsigned)std::min<int64_t>(blocks, 1024)), \
                                   dim3(256), lds_cells, st, nodes, M, queries, Q, out_idx, out_w, scratch_list,    \
                                   scratch_count, step);                                                            \
        } else                                                                                                      \
            hipLaunchKernelGGL(knn_main_kernel<KV>, dim3((unsigned)blocks), dim3(256), lds, st, nodes, M, queries,  \
                               Q, out_idx, out_w, scratch_list, scratch_count);                                     \
        break;
        ARAPGS_KNN_CASE(1) ARAPGS_KNN_CASE(2) ARAPGS_KNN_CASE(3) ARAPGS_KNN_CASE(4) ARAPGS_KNN_CASE(5)
        ARAPGS_KNN_CASE(6) ARAPGS_KNN_CASE(7) ARAPGS_KNN_CASE(8) ARAPGS_KNN_CASE(9) ARAPGS_KNN_CASE(10)
        ARAPGS_KNN_CASE(11) ARAPGS_KNN_CASE(12)
#undef ARAPGS_KNN_CASE
        default:
            return -1;
    }
    HIP_RET(hipGetLastError());
    hipLaunchKernelGGL(knn_fallback_kernel, dim3(1024), dim3(64), 0, st, nodes, M, queries, k, out_idx, out_w,
                       scratch_list, scratch_count);
    HIP_RET(hipGetLastError());
    return 0;
}

namespace {
int fps_wgs(int64_t N) { return (int)std::min<int64_t>((N + FPS_WG - 1) / FPS_WG, FPS_MAX_WGS + 1); }
size_t fps_slot_words(int64_t N) { return 2 * 4 * (size_t)fps_wgs(N) + 1; }
}  // namespace

size_t fps_workspace_bytes(int64_t N) {
    if (fps_wgs(N) > FPS_MAX_WGS) return 16 * (size_t)N;
    return 16 * (size_t)N + 8 * fps_slot_words(N) + sizeof(uint32_t) * radix_workspace_words(N) + 4096;
}

// Steps from which one launch pays for the sort that it needs (0.2 ms). In one
// launch and one a step: 1 step of 4k points 211 and 41 us, 24 steps 263 and 310;
// of 3M points 353 and 81, 491 and 595.
constexpr int FPS_FEW = 24;

// CUs that the stream's work may run on (a whole one's: all of the device's).
static int stream_cus(hipStream_t st) {
    uint32_t mask[64] = {};
    if (!st || hipExtStreamGetCUMask(st, 64, mask) != hipSuccess) {
        (void)hipGetLastError();
        return INT_MAX;
    }
    int n = 0;
    for (const uint32_t w : mask) n += __builtin_popcount(w);
    return n > 0 ? n : INT_MAX;
}

// In one launch for up to FPS_MAX_WGS workgroups' worth of points (3.1M); beyond
// that, on a stream of fewer CUs than workgroups (one a CU, which must all run at
// once), for few steps (FPS_FEW) and where the launch does not fit or gave up, one
// launch per step over all points. 1M points, 2048 nodes: 55.4 -> 7.6 ms (27.1 us a step over all
// points, 12.7 with one workgroup per CU; a single workgroup that read the few
// runs of points near the choice from memory took 12.4 us a step: one CU's loads
// in flight are too few).
int launch_fps(const float* pos, int64_t N, int m_steps, int* out, void* ws, unsigned long long* partial,
               int n_partial, unsigned int* counter, unsigned long long* best, int polls, hipStream_t st) {
    char* p = (char*)ws;
    const auto take = [&](size_t bytes) {
        char* r = p;
        p += (bytes + 255) & ~(size_t)255;
        return r;
    };
    const unsigned nb = (unsigned)((N + 255) / 256);
    hipLaunchKernelGGL(fps_clear_kernel, dim3(1), dim3(64), 0, st, best);
    hipLaunchKernelGGL(fps_first_kernel, dim3(std::min(nb, 512u)), dim3(256), 0, st, pos, N, best);
    const int wgs = fps_wgs(N);
    if (wgs <= FPS_MAX_WGS && m_steps >= FPS_FEW && polls > 0 && wgs <= stream_cus(st)) {
        uint32_t* keys = (uint32_t*)take(4 * (size_t)N);
        uint32_t* ids = (uint32_t*)take(4 * (size_t)N);
        uint32_t* keys_alt = (uint32_t*)take(4 * (size_t)N);
        uint32_t* ids_alt = (uint32_t*)take(4 * (size_t)N);
        float* box = (float*)take(64);
        uint32_t* mm = (uint32_t*)take(64);
        uint32_t* sort_ws = (uint32_t*)take(sizeof(uint32_t) * radix_workspace_words(N));
        const int64_t words = (int64_t)fps_slot_words(N);
        unsigned long long* slots = (unsigned long long*)take(8 * (size_t)words);
        int* failed = (int*)(slots + words - 1);
        int rc = launch_minmax(pos, N, mm, box, st);
        if (rc) return rc;
        hipLaunchKernelGGL(fps_keys_kernel, dim3(nb), dim3(256), 0, st, pos, N, box, keys, ids);
        rc = launch_radix_sort32(keys, ids, keys_alt, ids_alt, N, 30, sort_ws, st);
        if (rc) return rc;
        hipLaunchKernelGGL(fps_init_kernel, dim3(8), dim3(256), 0, st, pos, N, (float4*)nullptr, slots, words, best,
                           out, counter);
        HIP_RET(hipGetLastError());
        const uint32_t* cids = ids;
        void* args[] = {&pos, &N, &cids, &m_steps, &out, &slots, &polls, &failed};
        if (hipLaunchCooperativeKernel(reinterpret_cast<const void*>(fps_resident_kernel), dim3((unsigned)wgs),
                                       dim3(1024), args, 0, st) == hipSuccess) {
            int gave_up = 0;
            HIP_RET(hipMemcpyAsync(&gave_up, failed, sizeof(int), hipMemcpyDeviceToHost, st));
            HIP_RET(hipStreamSynchronize(st));
            if (!gave_up) return 0;
        } else {
            (void)hipGetLastError();
        }
    }
    float4* pts = (float4*)ws;
    hipLaunchKernelGGL(fps_init_kernel, dim3(std::min(nb, 2048u)), dim3(256), 0, st, pos, N, pts,
                       (unsigned long long*)nullptr, (int64_t)0, best, out, counter);
    for (int s = 0; s < m_steps; s++)
        hipLaunchKernelGGL(fps_step_kernel, dim3(std::min<unsigned>(n_partial, 256u)), dim3(1024), 0, st, pos, N, pts, s,
                           out, partial, counter);
    HIP_RET(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------- no-allocation KNN
// The scratch of arapgs_knn_noalloc: word 0 is the fallback count, words
// 64 .. 64 + KNN_NOALLOC_MAX_QUERIES - 1 the fallback list. Every GPU that
// loads the library holds its own copy until the process ends. In host code
// `scratch` names a host-side stand-in, not device memory: host code uses only
// the per-device address that hipGetSymbolAddress returned.
static __device__ __align__(256) uint32_t scratch[64 + KNN_NOALLOC_MAX_QUERIES];

namespace {
std::mutex g_scratch_mu;
uint32_t* g_scratch_ptr[KNN_NOALLOC_MAX_DEVICES] = {};
}  // namespace

int knn_noalloc_scratch(int device, uint32_t** out) {
    *out = nullptr;
    if (device < 0 || device >= KNN_NOALLOC_MAX_DEVICES) return -1;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        int cur = -1;
        HIP_RET(hipGetDevice(&cur));
        if (cur != device) return -1;  // the caller makes the device current
        void* p = nullptr;
        HIP_RET(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return -1;
        g_scratch_ptr[device] = static_cast<uint32_t*>(p);
    }
    *out = g_scratch_ptr[device];
    return 0;
}

}  // namespace arapgs
