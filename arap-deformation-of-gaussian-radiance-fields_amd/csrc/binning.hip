// Tile lists of a render (gfx950): the visible (view, Gaussian) records are
// sorted by depth, and the tiles of their rectangles, in that order, are sorted
// by tile id, all stably, so that every tile's list comes out ordered by (depth
// bits, record) as a stable sort of (tile << 32 | depth bits) keys would.
//
// A render of 3M Gaussians in 8 views at 1080p has 24M records and 300M tile
// instances, so the bytes and instructions of an instance are what it costs. The
// instances are never written unsorted: both kernels of the first pass (digit
// counts, then the scatter) take them from the sorted records, which lie in L2.
// The first pass sorts by the low half of the tile id and leaves the high half
// (one byte) with the record index; the second one leaves the record index
// only. Its workgroups do not cross a change of the low half, so the scanned
// counts of the second pass are the tiles' ranges. 15 bytes an instance in all,
// against 52 for emission, two passes over 32-bit (tile, record) pairs and a
// pass over the sorted keys for the ranges. Measured at that size: instances
// 6.9 -> 2.9 ms (counts 0.43, scatter 1.24, counts 0.29, scatter 0.82: ranking,
// some 65 vector instructions per instance, bounds the scatters), records 1.3 ->
// 1.1 ms (0.49 of it the random read of the rectangles). Tiles of 2048, 4096 and
// 8192 instances with 256 to 512 threads measured within 5%; 1024 threads 20%
// slower.
//
// A render of 100k Gaussians at 800 x 800 (313k instances) is launches: 36
// become 15 where the workgroups of a pass add up the counts themselves
// (FUSED_BLOCKS); with the blend 315 -> 204 us.
#include "binning.hpp"
#include "sort.hpp"

namespace arapgs {

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

constexpr int DIGITS = 256;

// Exclusive prefix of v over the workgroup; s holds a word per wave.
template <int THREADS>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s[wave] = x;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < wave; w++) before += s[w];
    __syncthreads();
    return before + x - v;
}

// A workgroup's stable scatter of up to THREADS * ITEMS elements by a digit of
// BITS bits: items are held wave by wave, 64 at a time in order (item it of lane
// l of wave w is element (w * ITEMS + it) * 64 + l). Ranks: lanes with equal
// digits found by one ballot per bit, counts per wave and digit in LDS.
template <int THREADS, int ITEMS, int BITS>
struct Ranker {
    static constexpr int WAVES = THREADS / 64;
    uint32_t count[WAVES][1 << BITS];
    uint32_t start[1 << BITS];  // first slot of a digit in the workgroup's sorted order
    uint32_t scan[WAVES];

    __device__ __forceinline__ void rank(const uint32_t (&digit)[ITEMS], const bool (&valid)[ITEMS],
                                         uint32_t (&slot)[ITEMS]) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for (int i = threadIdx.x; i < WAVES << BITS; i += THREADS) (&count[0][0])[i] = 0;
        __syncthreads();
        const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t dg = digit[it];
            const uint64_t ok = __ballot(valid[it]);
            uint32_t el = (uint32_t)ok, eh = (uint32_t)(ok >> 32);
#pragma unroll
            for (int b = 0; b < BITS; b++) {  // eq &= ~(ballot ^ own bit): one three-input instruction a half
                const uint32_t own = 0u - ((dg >> b) & 1u);
                const uint64_t bal = __ballot(own != 0u);
                el &= ~((uint32_t)bal ^ own);
                eh &= ~((uint32_t)(bal >> 32) ^ own);
            }
            const uint64_t eq = (uint64_t)eh << 32 | el;
            const uint32_t prev = valid[it] ? count[wave][dg] : 0u;
            slot[it] = prev + (uint32_t)__popcll(eq & below);
            __builtin_amdgcn_wave_barrier();
            // the highest lane of each digit publishes the new count
            if (valid[it] && (eq >> lane) == 1ull) count[wave][dg] = prev + (uint32_t)__popcll(eq);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        uint32_t total = 0;
        const int d = threadIdx.x;
        if (d < 1 << BITS)
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                const uint32_t c = count[w][d];
                count[w][d] = total;
                total += c;
            }
        const uint32_t first = block_scan<THREADS>(total, scan);
        if (d < 1 << BITS) start[d] = first;
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITEMS; it++)
            if (valid[it]) slot[it] += start[digit[it]] + count[wave][digit[it]];
    }
};

// First slot of every digit of this workgroup (into s_off, 1 << BITS of them).
// FUSED (up to FUSED_BLOCKS workgroups): hist is block-major and every workgroup
// adds the counts up for itself, which costs less than the three launches of a
// scan (FUSED_BLOCKS), and leaves its own starts in offs. Otherwise offs is the
// scan of the digit-major counts.
template <int THREADS, int BITS, bool FUSED>
__device__ __forceinline__ void digit_offsets(const uint32_t* __restrict__ hist, uint32_t* __restrict__ offs,
                                              uint32_t* s_off, uint32_t* s_scan) {
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    const uint32_t d = threadIdx.x;
    if constexpr (FUSED) {
        uint32_t before = 0, total = 0;
        if (d < (1u << BITS)) {
#pragma unroll 16
            for (uint32_t i = 0; i < nb; i++) {
                const uint32_t c = hist[(i << BITS) + d];
                before += i < b ? c : 0u;
                total += c;
            }
        }
        const uint32_t at = block_scan<THREADS>(total, s_scan) + before;
        if (d < (1u << BITS)) {
            s_off[d] = at;
            offs[(int64_t)d * nb + b] = at;
        }
    } else {
        for (uint32_t i = d; i < (1u << BITS); i += THREADS) s_off[i] = offs[(int64_t)i * nb + b];
    }
}

// Where a workgroup's count of digit d goes.
template <int BITS, bool FUSED>
__device__ __forceinline__ uint32_t& digit_count(uint32_t* __restrict__ hist, uint32_t d) {
    return FUSED ? hist[(blockIdx.x << BITS) + d] : hist[(int64_t)d * gridDim.x + blockIdx.x];
}

// ------------------------------------------------------------ records by depth
// Key of record gv: 0 where nothing is visible (depth 0), else its depth bits
// above the frame's smallest, from 1.
__device__ __forceinline__ uint32_t depth_key(uint32_t bits, uint32_t dmin) { return bits ? bits - dmin + 1u : 0u; }

// FIRST: the keys are made from the depths (and the values are the indices).
template <int THREADS, int ITEMS, bool FUSED, bool FIRST>
__global__ void __launch_bounds__(THREADS) record_hist_kernel(const uint32_t* __restrict__ keys, int64_t n,
                                                              uint32_t dmin, int shift, uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[DIGITS];
    for (int i = threadIdx.x; i < DIGITS; i += THREADS) h[i] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (THREADS * ITEMS);
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int64_t i = base + it * THREADS + threadIdx.x;
        if (i < n) {
            const uint32_t k = FIRST ? depth_key(keys[i], dmin) : keys[i];
            atomicAdd(&h[(k >> shift) & (DIGITS - 1)], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < DIGITS; i += THREADS) digit_count<8, FUSED>(hist, i) = h[i];
}

// LAST: only the values are written.
template <int THREADS, int ITEMS, bool FUSED, bool FIRST, bool LAST>
__global__ void __launch_bounds__(THREADS) record_scatter_kernel(const uint32_t* __restrict__ keys,
                                                                 const uint32_t* __restrict__ vals, int64_t n,
                                                                 uint32_t dmin, int shift,
                                                                 const uint32_t* __restrict__ hist,
                                                                 uint32_t* __restrict__ offs,
                                                                 uint32_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ vals_out) {
    __shared__ Ranker<THREADS, ITEMS, 8> R;
    __shared__ uint32_t s_off[DIGITS];
    __shared__ uint32_t s_key[THREADS * ITEMS];
    __shared__ uint32_t s_val[THREADS * ITEMS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t base = (int64_t)blockIdx.x * (THREADS * ITEMS);
    const int here = (int)min((int64_t)(THREADS * ITEMS), n - base);
    uint32_t key[ITEMS], val[ITEMS], digit[ITEMS], slot[ITEMS];
    bool valid[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int e = (wave * ITEMS + it) * 64 + lane;
        valid[it] = e < here;
        const int64_t at = base + min(e, here - 1);
        key[it] = FIRST ? depth_key(keys[at], dmin) : keys[at];
        val[it] = FIRST ? (uint32_t)at : vals[at];
        digit[it] = (key[it] >> shift) & (DIGITS - 1);
    }
    digit_offsets<THREADS, 8, FUSED>(hist, offs, s_off, R.scan);
    R.rank(digit, valid, slot);
#pragma unroll
    for (int it = 0; it < ITEMS; it++)
        if (valid[it]) {
            s_key[slot[it]] = key[it];
            s_val[slot[it]] = val[it];
        }
    __syncthreads();
    for (int i = threadIdx.x; i < here; i += THREADS) {
        const uint32_t k = s_key[i], dg = (k >> shift) & (DIGITS - 1);
        const uint32_t dst = s_off[dg] + (uint32_t)i - R.start[dg];
        if (!LAST) keys_out[dst] = k;
        vals_out[dst] = s_val[i];
    }
}

// ------------------------------------------------------ the sorted records' tiles
constexpr int REC_THREADS = 256, REC_ITEMS = 8, REC_TILE = REC_THREADS * REC_ITEMS;

// Rectangles of the visible records in depth order (the one random read of the
// pipeline) and the instance counts of every REC_TILE of them.
__global__ void __launch_bounds__(REC_THREADS) record_gather_kernel(const uint32_t* __restrict__ recs, int64_t n,
                                                                    const TileRect* __restrict__ rects,
                                                                    TileRect* __restrict__ sorted,
                                                                    uint32_t* __restrict__ sums) {
    __shared__ uint32_t s[REC_THREADS / 64];
    const int64_t base = (int64_t)blockIdx.x * REC_TILE;
    TileRect r[REC_ITEMS];
    uint32_t total = 0;
#pragma unroll
    for (int it = 0; it < REC_ITEMS; it++) {
        const int64_t i = base + it * REC_THREADS + threadIdx.x;
        r[it] = i < n ? rects[recs[i]] : TileRect{0, 0};
        total += r[it].area;
    }
#pragma unroll
    for (int it = 0; it < REC_ITEMS; it++) {
        const int64_t i = base + it * REC_THREADS + threadIdx.x;
        if (i < n) sorted[i] = r[it];
    }
    for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = total;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// First instance of every sorted record, and the record that holds the first
// instance of every `tile` instances (starts[nb] = the last record). sums: the
// workgroups' instance counts, scanned or (few of them) as they are.
__global__ void __launch_bounds__(REC_THREADS) record_starts_kernel(const TileRect* __restrict__ sorted, int64_t n,
                                                                    const uint32_t* __restrict__ sums, bool scanned,
                                                                    uint32_t tile, uint32_t nb, uint32_t* __restrict__ first,
                                                                    uint32_t* __restrict__ starts) {
    __shared__ uint32_t s[REC_THREADS / 64];
    const int64_t base = (int64_t)blockIdx.x * REC_TILE + (int64_t)threadIdx.x * REC_ITEMS;
    uint32_t area[REC_ITEMS], total = 0;
#pragma unroll
    for (int it = 0; it < REC_ITEMS; it++) {
        area[it] = base + it < n ? sorted[base + it].area : 0u;
        total += area[it];
    }
    uint32_t before = scanned && threadIdx.x == 0 ? sums[blockIdx.x] : 0u;
    if (!scanned)
        for (uint32_t i = threadIdx.x; i < blockIdx.x; i += REC_THREADS) before += sums[i];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
    uint32_t at = block_scan<REC_THREADS>(total, s);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = before;
    __syncthreads();
    at += s[0] + s[1] + s[2] + s[3];
#pragma unroll
    for (int it = 0; it < REC_ITEMS; it++) {
        if (base + it >= n) break;
        first[base + it] = at;
        for (uint32_t k = (at + tile - 1) / tile; (uint64_t)k * tile < (uint64_t)at + area[it]; k++)
            starts[k] = (uint32_t)(base + it);
        at += area[it];
        if (base + it == n - 1) starts[nb] = (uint32_t)(n - 1);
    }
}

// The records of a workgroup's `here` instances from instance `base` on, as a
// bit per instance that starts a record after r0 = the record of the first one
// (every record has an instance, so no two start at one) and a prefix count per
// 64 of them: the record of an instance is r0 + the bits up to it.
template <int THREADS, int ITEMS>
struct Starts {
    static constexpr int WORDS = THREADS * ITEMS / 64;
    unsigned long long bits[WORDS];
    uint32_t before[WORDS];

    __device__ __forceinline__ void make(const uint32_t* __restrict__ first, uint32_t r0, uint32_t r1, uint32_t base,
                                         int here, uint32_t* s_scan) {
        for (int i = threadIdx.x; i < WORDS; i += THREADS) bits[i] = 0ull;
        __syncthreads();
        for (uint32_t r = r0 + 1 + threadIdx.x; r <= r1; r += THREADS) {
            const uint32_t at = first[r] - base;
            if (at < (uint32_t)here) atomicOr(&bits[at >> 6], 1ull << (at & 63));
        }
        __syncthreads();
        const uint32_t c = threadIdx.x < WORDS ? (uint32_t)__popcll(bits[threadIdx.x]) : 0u;
        const uint32_t at = block_scan<THREADS>(c, s_scan);
        if (threadIdx.x < WORDS) before[threadIdx.x] = at;
        __syncthreads();
    }
    // of instance word * 64 + lane, as an index from r0
    __device__ __forceinline__ uint32_t record(int word, int lane) const {
        const unsigned long long b = bits[word];
        return before[word] + (uint32_t)__popcll(b & (~0ull >> (63 - lane)));
    }
};

// Tile of instance q of a rectangle. q < 65536, so (q + 1/2) / w is 2^-17 of
// itself or more away from a whole number, and the reciprocal's last bit does
// not matter.
__device__ __forceinline__ uint32_t tile_of(const TileRect& r, uint32_t q, uint32_t gx) {
    const uint32_t w = r.base_w & 0xffffu;
    const uint32_t y = (uint32_t)(((float)q + 0.5f) * __builtin_amdgcn_rcpf((float)w));
    return (r.base_w >> 16) + y * gx + (q - y * w);
}

template <int THREADS, int ITEMS, int BITS, bool FUSED>
__global__ void __launch_bounds__(THREADS) instance_hist_kernel(const TileRect* __restrict__ sorted,
                                                                const uint32_t* __restrict__ first,
                                                                const uint32_t* __restrict__ starts, uint32_t n,
                                                                uint32_t gx, uint32_t* __restrict__ hist) {
    constexpr uint32_t MASK = (1u << BITS) - 1u;
    __shared__ Starts<THREADS, ITEMS> S;
    __shared__ uint32_t s_scan[THREADS / 64];
    __shared__ uint32_t h[1 << BITS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t i = threadIdx.x; i <= MASK; i += THREADS) h[i] = 0;
    const uint32_t base = blockIdx.x * (uint32_t)(THREADS * ITEMS);
    const int here = (int)min((uint32_t)(THREADS * ITEMS), n - base);
    const uint32_t r0 = starts[blockIdx.x];
    S.make(first, r0, starts[blockIdx.x + 1], base, here, s_scan);
    uint32_t tile[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int word = wave * ITEMS + it;
        const uint32_t e = min((uint32_t)(word * 64 + lane), (uint32_t)here - 1u);
        const uint32_t r = r0 + S.record((int)(e >> 6), (int)(e & 63));
        tile[it] = tile_of(sorted[r], base + e - first[r], gx);
    }
#pragma unroll
    for (int it = 0; it < ITEMS; it++)
        if ((wave * ITEMS + it) * 64 + lane < here) atomicAdd(&h[tile[it] & MASK], 1u);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i <= MASK; i += THREADS) digit_count<BITS, FUSED>(hist, i) = h[i];
}

// The first pass: instances enumerated, sorted by the low BITS of the tile; the
// rest of the tile id goes to rest[] (null: there is none).
template <int THREADS, int ITEMS, int BITS, bool FUSED>
__global__ void __launch_bounds__(THREADS) instance_scatter_kernel(
    const TileRect* __restrict__ sorted, const uint32_t* __restrict__ first, const uint32_t* __restrict__ starts,
    const uint32_t* __restrict__ recs, uint32_t n, uint32_t gx, const uint32_t* __restrict__ hist,
    uint32_t* __restrict__ offs, uint8_t* __restrict__ rest, uint32_t* __restrict__ vals) {
    constexpr uint32_t MASK = (1u << BITS) - 1u;
    __shared__ Ranker<THREADS, ITEMS, BITS> R;
    __shared__ Starts<THREADS, ITEMS> S;
    __shared__ uint32_t s_off[1 << BITS];
    __shared__ uint32_t s_val[THREADS * ITEMS];
    __shared__ uint16_t s_tile[THREADS * ITEMS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t base = blockIdx.x * (uint32_t)(THREADS * ITEMS);
    const int here = (int)min((uint32_t)(THREADS * ITEMS), n - base);
    const uint32_t r0 = starts[blockIdx.x];
    S.make(first, r0, starts[blockIdx.x + 1], base, here, R.scan);
    uint32_t tile[ITEMS], val[ITEMS], digit[ITEMS], slot[ITEMS];
    bool valid[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int word = wave * ITEMS + it;
        const uint32_t e = min((uint32_t)(word * 64 + lane), (uint32_t)here - 1u);
        valid[it] = word * 64 + lane < here;
        const uint32_t r = r0 + S.record((int)(e >> 6), (int)(e & 63));
        tile[it] = tile_of(sorted[r], base + e - first[r], gx);
        val[it] = recs[r];
        digit[it] = tile[it] & MASK;
    }
    digit_offsets<THREADS, BITS, FUSED>(hist, offs, s_off, R.scan);
    R.rank(digit, valid, slot);
#pragma unroll
    for (int it = 0; it < ITEMS; it++)
        if (valid[it]) {
            s_tile[slot[it]] = (uint16_t)tile[it];
            s_val[slot[it]] = val[it];
        }
    __syncthreads();
    for (int i = threadIdx.x; i < here; i += THREADS) {
        const uint32_t t = s_tile[i], dg = t & MASK;
        const uint32_t dst = s_off[dg] + (uint32_t)i - R.start[dg];
        if (rest) rest[dst] = (uint8_t)(t >> BITS);
        vals[dst] = s_val[i];
    }
}

// First workgroup of the second pass for every value d of the low digit (values
// start at offs[d * nb1]): each value's instances fill whole workgroups.
__global__ void __launch_bounds__(DIGITS) second_blocks_kernel(const uint32_t* __restrict__ offs, uint32_t nb1,
                                                               uint32_t n, uint32_t values, uint32_t tile,
                                                               uint32_t* __restrict__ value_at,
                                                               uint32_t* __restrict__ block_at) {
    __shared__ uint32_t s[DIGITS / 64];
    const uint32_t d = threadIdx.x;
    const uint32_t a = d < values ? offs[(int64_t)d * nb1] : n;
    const uint32_t b = d + 1 < values ? offs[(int64_t)(d + 1) * nb1] : n;
    const uint32_t blocks = (b - a + tile - 1) / tile;
    const uint32_t at = block_scan<DIGITS>(blocks, s);
    value_at[d] = a;
    block_at[d] = at;
    if (d == DIGITS - 1) {
        value_at[DIGITS] = n;
        block_at[DIGITS] = at + blocks;
    }
}

// This workgroup's instances [beg, beg + here) of the second pass (here = 0:
// none). The search runs on scalar loads; one compare a thread and a word in LDS
// measured slower (it takes two barriers).
template <int TILE>
__device__ __forceinline__ int second_range(const uint32_t* __restrict__ value_at, const uint32_t* __restrict__ block_at,
                                            uint32_t& beg) {
    beg = 0;
    if (blockIdx.x >= block_at[DIGITS]) return 0;
    int lo = 0;  // the last value whose first workgroup is <= this one (values without instances have none)
#pragma unroll
    for (int step = DIGITS / 2; step >= 1; step >>= 1)
        if (block_at[lo + step] <= blockIdx.x) lo += step;
    beg = value_at[lo] + (blockIdx.x - block_at[lo]) * TILE;
    return (int)min((uint32_t)TILE, value_at[lo + 1] - beg);
}

template <int THREADS, int ITEMS, int BITS, bool FUSED>
__global__ void __launch_bounds__(THREADS) second_hist_kernel(const uint8_t* __restrict__ rest,
                                                              const uint32_t* __restrict__ value_at,
                                                              const uint32_t* __restrict__ block_at,
                                                              uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[1 << BITS];
    for (int i = threadIdx.x; i < 1 << BITS; i += THREADS) h[i] = 0;
    __syncthreads();
    uint32_t beg;
    const int here = second_range<THREADS * ITEMS>(value_at, block_at, beg);
    if (here > 0) {  // uniform
        uint32_t digit[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) digit[it] = rest[beg + (uint32_t)min(it * THREADS + (int)threadIdx.x, here - 1)];
#pragma unroll
        for (int it = 0; it < ITEMS; it++)
            if (it * THREADS + (int)threadIdx.x < here) atomicAdd(&h[digit[it]], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 1 << BITS; i += THREADS) digit_count<BITS, FUSED>(hist, i) = h[i];
}

template <int THREADS, int ITEMS, int BITS, bool FUSED>
__global__ void __launch_bounds__(THREADS) second_scatter_kernel(const uint8_t* __restrict__ rest,
                                                                 const uint32_t* __restrict__ vals,
                                                                 const uint32_t* __restrict__ value_at,
                                                                 const uint32_t* __restrict__ block_at,
                                                                 const uint32_t* __restrict__ hist,
                                                                 uint32_t* __restrict__ offs,
                                                                 uint32_t* __restrict__ vals_out) {
    __shared__ Ranker<THREADS, ITEMS, BITS> R;
    __shared__ uint32_t s_off[1 << BITS];
    __shared__ uint32_t s_val[THREADS * ITEMS];
    __shared__ uint8_t s_dig[THREADS * ITEMS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t beg;
    const int here = second_range<THREADS * ITEMS>(value_at, block_at, beg);
    digit_offsets<THREADS, BITS, FUSED>(hist, offs, s_off, R.scan);
    if (here == 0) return;  // uniform
    uint32_t val[ITEMS], digit[ITEMS], slot[ITEMS];
    bool valid[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int e = (wave * ITEMS + it) * 64 + lane;
        valid[it] = e < here;
        const uint32_t at = beg + (uint32_t)min(e, here - 1);
        digit[it] = rest[at];
        val[it] = vals[at];
    }
    R.rank(digit, valid, slot);
#pragma unroll
    for (int it = 0; it < ITEMS; it++)
        if (valid[it]) {
            s_dig[slot[it]] = (uint8_t)digit[it];
            s_val[slot[it]] = val[it];
        }
    __syncthreads();
    for (int i = threadIdx.x; i < here; i += THREADS) {
        const uint32_t dg = s_dig[i];
        vals_out[s_off[dg] + (uint32_t)i - R.start[dg]] = s_val[i];
    }
}

// Range of tile (hi, lo): from the second pass's scanned counts (hi's run begins,
// for the low value lo, at offs[hi][first workgroup of lo]), or from the first
// pass's where it is the only one (bits_hi = 0).
__global__ void __launch_bounds__(256) tile_ranges_kernel(const uint32_t* __restrict__ offs, uint32_t nb,
                                                          const uint32_t* __restrict__ block_at, int bits_lo,
                                                          int bits_hi, uint32_t n, uint32_t tiles,
                                                          uint2* __restrict__ ranges) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= tiles) return;
    const auto start = [&](uint32_t hi, uint32_t lo) {  // lo may be one past the last value
        if (bits_hi == 0) return lo < (1u << bits_lo) ? offs[(int64_t)lo * nb] : n;
        const uint64_t at = (uint64_t)hi * nb + (lo < (1u << bits_lo) ? block_at[lo] : nb);
        return at < ((uint64_t)nb << bits_hi) ? offs[at] : n;
    };
    const uint32_t lo = t & ((1u << bits_lo) - 1u), hi = t >> bits_lo;
    const uint2 r = make_uint2(start(hi, lo), start(hi, lo + 1));
    ranges[t] = r.x < r.y ? r : make_uint2(0u, 0u);  // an empty tile's range is (0, 0)
}

// No instances: empty ranges.
__global__ void __launch_bounds__(256) empty_ranges_kernel(uint32_t tiles, uint2* __restrict__ ranges) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < tiles) ranges[t] = make_uint2(0u, 0u);
}

// Workgroup shapes of the sorts: small ones fill the chip with few elements,
// large ones move longer runs of a digit and scan fewer counts. Whole renders with
// small and with large workgroups: 3.2M instances 261 and 301 us, 11.8M 430 and
// 451, 18M 619 and 599 (the records in small ones), 93M 2.27 and 1.91 ms; 2M
// records 636 and 645 us, 4M 1058 and 1029.
constexpr int S_THREADS = 256, S_ITEMS = 8, L_THREADS = 512, L_ITEMS = 16;
constexpr int64_t LARGE_RECORDS = 2 << 20, LARGE_INSTANCES = 16 << 20;
// Workgroups that add up the others' counts read 1 KB for each of them, 16 loads
// in flight: at 153 workgroups the scatter grows from 10 to 14 us, and the three
// launches of a scan (13 us) go; past about 400 the sums cost more than those.
constexpr unsigned FUSED_BLOCKS = 256;
inline uint32_t sort_tile(bool large) { return large ? L_THREADS * L_ITEMS : S_THREADS * S_ITEMS; }

// f(threads, items, fused) with the shape for nb workgroups.
template <int V>
struct Int {
    static constexpr int value = V;
};
template <typename F>
int with_shape(bool large, unsigned nb, F f) {
    if (large) return f(Int<L_THREADS>{}, Int<L_ITEMS>{}, Int<0>{});
    return nb <= FUSED_BLOCKS ? f(Int<S_THREADS>{}, Int<S_ITEMS>{}, Int<1>{}) : f(Int<S_THREADS>{}, Int<S_ITEMS>{}, Int<0>{});
}
// f(bits) for a digit of 5 to 8 bits.
template <typename F>
int with_bits(int bits, F f) {
    return bits <= 5 ? f(Int<5>{}) : bits == 6 ? f(Int<6>{}) : bits == 7 ? f(Int<7>{}) : f(Int<8>{});
}

struct Carve {
    char* p;
    size_t used = 0;
    void* take(size_t bytes) {
        void* r = p ? p + used : nullptr;
        used += (bytes + 255) & ~(size_t)255;
        return r;
    }
};

struct RecordWs {
    uint32_t *keys[2], *vals[2], *hist, *offs, *scan, *sums, *sums_at, *first;
    TileRect* sorted;
    RecordWs(Carve c, int64_t PV, size_t* bytes = nullptr) {
        const size_t n = (size_t)std::max<int64_t>(PV, 1), nb = nblk((int64_t)n, (int)sort_tile((int64_t)n >= LARGE_RECORDS));
        for (int i = 0; i < 2; i++) keys[i] = (uint32_t*)c.take(4 * n);
        for (int i = 0; i < 2; i++) vals[i] = (uint32_t*)c.take(4 * n);
        hist = (uint32_t*)c.take(4 * DIGITS * nb);
        offs = (uint32_t*)c.take(4 * DIGITS * nb);
        sums = (uint32_t*)c.take(4 * (n / REC_TILE + 2));
        sums_at = (uint32_t*)c.take(4 * (n / REC_TILE + 2));
        scan = (uint32_t*)c.take(4 * (scan_workspace_words((int64_t)std::max<size_t>(DIGITS * nb, n / REC_TILE + 2)) + 64));
        first = (uint32_t*)c.take(4 * n);
        sorted = (TileRect*)c.take(sizeof(TileRect) * n);
        if (bytes) *bytes = c.used;
    }
};

struct InstanceWs {
    uint32_t *vals[2], *starts, *hist, *offs, *scan, *value_at, *block_at;
    uint8_t* rest;
    uint32_t nb1;
    InstanceWs(Carve c, int64_t n, size_t* bytes = nullptr) {
        const int64_t m = std::max<int64_t>(n, 1);
        const uint32_t tile = sort_tile(m >= LARGE_INSTANCES);
        nb1 = nblk(m, (int)tile);
        const uint32_t nb2 = nb1 + DIGITS;  // at most, for the second pass
        for (int i = 0; i < 2; i++) vals[i] = (uint32_t*)c.take(4 * (size_t)m);
        rest = (uint8_t*)c.take((size_t)m);
        starts = (uint32_t*)c.take(4 * ((size_t)nb1 + 1));
        hist = (uint32_t*)c.take(4 * DIGITS * (size_t)nb2);
        offs = (uint32_t*)c.take(4 * DIGITS * (size_t)nb2);
        scan = (uint32_t*)c.take(4 * (scan_workspace_words(DIGITS * (int64_t)nb2) + 64));
        value_at = (uint32_t*)c.take(4 * (DIGITS + 1));
        block_at = (uint32_t*)c.take(4 * (DIGITS + 1));
        if (bytes) *bytes = c.used;
    }
};

int sort_records(const BinInput& in, RecordWs& W, const uint32_t** recs, hipStream_t st) {
    const int64_t n = in.records;
    const bool large = n >= LARGE_RECORDS;
    const unsigned nb = nblk(n, (int)sort_tile(large));
    const uint32_t* keys = reinterpret_cast<const uint32_t*>(in.depth);
    const uint32_t* vals = nullptr;
    const int passes = (in.dbits + 7) / 8;
    const int rc = with_shape(large, nb, [&](auto t, auto i, auto fused) -> int {
        constexpr int T = decltype(t)::value, I = decltype(i)::value;
        constexpr bool F = decltype(fused)::value != 0;
        for (int p = 0; p < passes; p++) {
            const int shift = 8 * p;
            const bool last = p == passes - 1;
            uint32_t *ko = W.keys[p & 1], *vo = W.vals[p & 1];
            const auto count = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(nb), dim3(T), 0, st, keys, n, in.dmin, shift, W.hist);
            };
            const auto move = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(nb), dim3(T), 0, st, keys, vals, n, in.dmin, shift,
                                   (const uint32_t*)W.hist, W.offs, ko, vo);
            };
            if (p == 0) count(record_hist_kernel<T, I, F, true>);
            else count(record_hist_kernel<T, I, F, false>);
            if (!F) {
                const int e = launch_exclusive_scan(W.hist, (int64_t)DIGITS * nb, W.offs, nullptr, W.scan, st);
                if (e) return e;
            }
            if (p == 0 && last) move(record_scatter_kernel<T, I, F, true, true>);
            else if (p == 0) move(record_scatter_kernel<T, I, F, true, false>);
            else if (last) move(record_scatter_kernel<T, I, F, false, true>);
            else move(record_scatter_kernel<T, I, F, false, false>);
            keys = ko;
            vals = vo;
        }
        return 0;
    });
    *recs = vals + (n - in.visible);  // nothing-visible records come first
    if (rc) return rc;
    HIP_RET(hipGetLastError());
    return 0;
}

// The instances by the low `lo` bits of their tile, then (hi > 0) by the others.
int sort_instances(const BinInput& in, const RecordWs& R, const uint32_t* recs, InstanceWs& W, int lo, int hi,
                   const uint32_t** vals, uint2* ranges, hipStream_t st) {
    const uint32_t n = in.instances, nb1 = W.nb1, nb2 = nb1 + (1u << lo);
    const bool large = n >= LARGE_INSTANCES;
    int rc = with_shape(large, nb1, [&](auto t, auto i, auto fused) {
        return with_bits(lo, [&](auto bits) -> int {
            constexpr int T = decltype(t)::value, I = decltype(i)::value, B = decltype(bits)::value;
            constexpr bool F = decltype(fused)::value != 0;
            hipLaunchKernelGGL((instance_hist_kernel<T, I, B, F>), dim3(nb1), dim3(T), 0, st, R.sorted, R.first, W.starts,
                               n, (uint32_t)in.gx, W.hist);
            if (!F) {
                const int e = launch_exclusive_scan(W.hist, (int64_t)nb1 << lo, W.offs, nullptr, W.scan, st);
                if (e) return e;
            }
            hipLaunchKernelGGL((instance_scatter_kernel<T, I, B, F>), dim3(nb1), dim3(T), 0, st, R.sorted, R.first,
                               W.starts, recs, n, (uint32_t)in.gx, W.hist, W.offs, hi ? W.rest : nullptr, W.vals[0]);
            return 0;
        });
    });
    if (rc) return rc;
    *vals = W.vals[0];
    if (hi) {
        hipLaunchKernelGGL(second_blocks_kernel, dim3(1), dim3(DIGITS), 0, st, W.offs, nb1, n, 1u << lo,
                           sort_tile(large), W.value_at, W.block_at);
        rc = with_shape(large, nb2, [&](auto t, auto i, auto fused) {
            return with_bits(hi, [&](auto bits) -> int {
                constexpr int T = decltype(t)::value, I = decltype(i)::value, B = decltype(bits)::value;
                constexpr bool F = decltype(fused)::value != 0;
                hipLaunchKernelGGL((second_hist_kernel<T, I, B, F>), dim3(nb2), dim3(T), 0, st, W.rest, W.value_at,
                                   W.block_at, W.hist);
                if (!F) {
                    const int e = launch_exclusive_scan(W.hist, (int64_t)nb2 << hi, W.offs, nullptr, W.scan, st);
                    if (e) return e;
                }
                hipLaunchKernelGGL((second_scatter_kernel<T, I, B, F>), dim3(nb2), dim3(T), 0, st, W.rest, W.vals[0],
                                   W.value_at, W.block_at, W.hist, W.offs, W.vals[1]);
                return 0;
            });
        });
        if (rc) return rc;
        *vals = W.vals[1];
    }
    hipLaunchKernelGGL(tile_ranges_kernel, dim3(nblk(in.tiles, 256)), dim3(256), 0, st, (const uint32_t*)W.offs,
                       hi ? nb2 : nb1, (const uint32_t*)W.block_at, lo, hi, n, (uint32_t)in.tiles, ranges);
    HIP_RET(hipGetLastError());
    return 0;
}

}  // namespace

size_t bin_record_bytes(int64_t records) {
    size_t bytes = 0;
    RecordWs(Carve{nullptr}, records, &bytes);
    return bytes;
}

size_t bin_instance_bytes(int64_t instances) {
    size_t bytes = 0;
    InstanceWs(Carve{nullptr}, instances, &bytes);
    return bytes;
}

int launch_binning(const BinInput& in, void* rec_ws, void* inst_ws, const uint32_t** vals, uint2* ranges,
                   hipStream_t st) {
    *vals = (const uint32_t*)inst_ws;
    if (in.instances == 0 || in.visible == 0) {
        hipLaunchKernelGGL(empty_ranges_kernel, dim3(nblk(in.tiles, 256)), dim3(256), 0, st, (uint32_t)in.tiles, ranges);
        HIP_RET(hipGetLastError());
        return 0;
    }
    RecordWs R(Carve{(char*)rec_ws}, in.records);
    InstanceWs W(Carve{(char*)inst_ws}, in.instances);
    const uint32_t* recs = nullptr;
    int rc = sort_records(in, R, &recs, st);
    if (rc) return rc;
    const uint32_t tile = sort_tile(in.instances >= LARGE_INSTANCES);
    const int64_t nv = in.visible;
    const unsigned nr = nblk(nv, REC_TILE);
    hipLaunchKernelGGL(record_gather_kernel, dim3(nr), dim3(REC_THREADS), 0, st, recs, nv, in.rects, R.sorted, R.sums);
    const bool scanned = nr > FUSED_BLOCKS;
    if (scanned && (rc = launch_exclusive_scan(R.sums, nr, R.sums_at, nullptr, R.scan, st))) return rc;
    hipLaunchKernelGGL(record_starts_kernel, dim3(nr), dim3(REC_THREADS), 0, st, (const TileRect*)R.sorted, nv,
                       (const uint32_t*)(scanned ? R.sums_at : R.sums), scanned, tile, W.nb1, R.first, W.starts);
    HIP_RET(hipGetLastError());
    int bits = 1;
    while ((1ll << bits) < in.tiles) bits++;
    // one pass up to 8 bits; else halves of at least 5 bits
    const int lo = bits <= 8 ? std::max(bits, 5) : std::max((bits + 1) / 2, bits - 8);
    const int hi = bits <= 8 ? 0 : std::max(bits - lo, 5);
    return sort_instances(in, R, recs, W, lo, hi, vals, ranges, st);
}

}  // namespace arapgs
