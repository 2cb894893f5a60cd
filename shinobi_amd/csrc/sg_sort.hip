// sg_sort.hip -- stable LSD radix sort of (key, value) pairs and a prefix
// scan for gfx950, both reduce-then-scan (no inter-block waiting).
//
// Sort (semantics of chag::pp::sort as driven by src/Utils/Sort.cu:28-56),
// per pass over tiles of 4096 or 1024 keys:
//   up     per-tile digit counts -> counts[digit][tile]
//   scan   one block per digit: exclusive scan of its row, and its total
//   down   scans the digit totals into bases, ranks the tile's keys per digit
//          with wave64 ballot matching (items in tile order, so the pass is
//          stable), stages the tile in LDS in digit order and writes every
//          digit run contiguously
// Only ceil(key_bits / radix_bits) passes run (the reference sorts 32-bit
// keys two bits at a time, 48 launches).
//
// Scan (src/Utils/Scan.h:35-68): block sums, one-block scan of the sums,
// then each block rescans its tile from its offset.
#include <algorithm>

#include "sg_device.hpp"
#include "sg_kernels.hpp"

namespace sg {

// Keys per thread.  A tile of 16 x 256 keys writes its digit runs in whole
// cache lines; a small sort then has few tiles, and each waits for 16 ranking
// rounds in a row, so sorts of up to kSmallSort pairs take 4 keys per thread.
// (26,000 pairs: k_sort_down 11.4 -> 6.5 us a pass, k_sort_up 4.1 -> 2.4; 546,000
// pairs of a capacity of a million and more: 11.2 -> 7.8 and 4.7 -> 4.3; at
// 2.46 M pairs the smaller tiles were 10 us slower.)  The line is drawn on the
// capacity, which a grid's build leaves at about twice its pairs.
constexpr int kSortItems = 16, kSmallItems = 4;
constexpr uint32_t kSmallSort = 1u << 21;
// Up to this many tiles a tile's digit offsets are folded by the downsweep
// itself from counts stored [tile][digit] (one row of them per tile before
// it), and the scan launch between the sweeps, 3 us and a gap, falls away.
constexpr uint32_t kFoldTiles = 64;

static int sort_items(uint32_t cap) { return cap <= kSmallSort ? kSmallItems : kSortItems; }

int sort_passes(int key_bits, int radix_bits) {
    if (key_bits < 1) key_bits = 1;
    return (key_bits + radix_bits - 1) / radix_bits;
}

static size_t sort_tiles(uint32_t cap, int items) {
    const size_t tile = (size_t)kBlock * items;
    return ((size_t)cap + tile - 1) / tile;
}

uint32_t multi_sort_tiles(uint32_t cap) { return (uint32_t)sort_tiles(cap, kSortItems); }

size_t sort_scratch_words(uint32_t cap, int key_bits, int radix_bits) {
    const size_t R = (size_t)1 << radix_bits;
    const size_t passes = (size_t)sort_passes(key_bits, radix_bits);
    // a larger capacity never needs less: scratch grown by a larger call serves
    // a smaller one under capture
    size_t tiles = sort_tiles(cap, sort_items(cap));
    if (cap > kSmallSort) tiles = std::max(tiles, sort_tiles(kSmallSort, kSmallItems));
    size_t w = passes * R + R * (tiles + 1);
    return (w + 3) & ~(size_t)3;   // 16-byte multiple
}

// per-tile digit counts of one pass -> counts[d * T + tile], with FOLD
// counts[tile * R + d].  Each thread counts ITEMS consecutive keys and adds runs of equal digits with one LDS
// atomic, so runs of equal keys (cell-ordered emission) do not serialise.
// (the kernels are bodies taking the tile / digit index `bid`, called by
// the single-sort kernels with blockIdx.x and by the multi-grid kernels
// with the block's index within its grid)
template <int RB, int ITEMS, bool FOLD>
SG_D void sort_up_body(const uint32_t* __restrict__ keys, const uint32_t* d_n, uint32_t cap, int shift,
                       uint32_t* __restrict__ counts, uint32_t T, uint32_t bid) {
    constexpr int R = 1 << RB;
    __shared__ uint32_t s[R];
    const uint32_t n = min(*d_n, cap);
    const uint32_t base = bid * (kBlock * ITEMS);
    if (base >= n) return;
    for (int i = threadIdx.x; i < R; i += kBlock) s[i] = 0;
    __syncthreads();
    const uint32_t i0 = base + threadIdx.x * ITEMS;
    uint32_t k[ITEMS];
    if (i0 + ITEMS <= n) {
#pragma unroll
        for (int q = 0; q < ITEMS / 4; ++q) {
            const uint4 v = reinterpret_cast<const uint4*>(keys + i0)[q];
            k[4 * q] = v.x; k[4 * q + 1] = v.y; k[4 * q + 2] = v.z; k[4 * q + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) k[j] = i0 + j < n ? keys[i0 + j] : 0u;
    }
    const uint32_t m = i0 < n ? min((uint32_t)ITEMS, n - i0) : 0u;
    uint32_t rd = 0, rc = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        if ((uint32_t)j < m) {
            const uint32_t d = (k[j] >> shift) & (R - 1);
            if (rc && d != rd) {
                atomicAdd(&s[rd], rc);
                rc = 0;
            }
            rd = d;
            ++rc;
        }
    }
    if (rc) atomicAdd(&s[rd], rc);
    __syncthreads();
    for (int d = threadIdx.x; d < R; d += kBlock) counts[FOLD ? (size_t)bid * R + d : (size_t)d * T + bid] = s[d];
}

template <int RB, int ITEMS, bool FOLD>
__global__ __launch_bounds__(kBlock) void k_sort_up(const uint32_t* __restrict__ keys, const uint32_t* d_n,
                                                    uint32_t cap, int shift, uint32_t* __restrict__ counts,
                                                    uint32_t T) {
    sort_up_body<RB, ITEMS, FOLD>(keys, d_n, cap, shift, counts, T, blockIdx.x);
}

// one block per digit d: counts[d][t] -> sum over t' < t (in place), and
// totals[d] = the digit's count over all tiles
template <int RB, int ITEMS>
SG_D void sort_scan_body(const uint32_t* d_n, uint32_t cap, uint32_t* __restrict__ totals,
                         uint32_t* __restrict__ counts, uint32_t T, uint32_t bid) {
    __shared__ uint32_t s_scan[kBlock / 64];
    const uint32_t n = min(*d_n, cap);
    const uint32_t tiles = (n + kBlock * ITEMS - 1) / (kBlock * ITEMS);
    const uint32_t d = bid;
    uint32_t run = 0;
    uint32_t* row = counts + (size_t)d * T;
    // chunks of 256*8 tiles: each thread scans 8 consecutive values
    for (uint32_t c0 = 0; c0 < tiles; c0 += kBlock * 8) {
        const uint32_t t0 = c0 + threadIdx.x * 8;
        uint32_t v[8], sum = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            v[k] = t0 + k < tiles ? row[t0 + k] : 0u;
            sum += v[k];
        }
        uint32_t tot;
        uint32_t pre = run + block_excl_scan<kBlock / 64>(sum, &tot, s_scan);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (t0 + k < tiles) row[t0 + k] = pre;
            pre += v[k];
        }
        run += tot;
    }
    if (threadIdx.x == 0) totals[d] = run;
}

template <int RB, int ITEMS>
__global__ __launch_bounds__(kBlock) void k_sort_scan(const uint32_t* d_n, uint32_t cap,
                                                      uint32_t* __restrict__ totals,
                                                      uint32_t* __restrict__ counts, uint32_t T) {
    sort_scan_body<RB, ITEMS>(d_n, cap, totals, counts, T, blockIdx.x);
}

template <int RB, int ITEMS, bool FOLD>
SG_D void sort_down_body(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                         uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, const uint32_t* d_n,
                         uint32_t cap, int shift, const uint32_t* __restrict__ totals,
                         const uint32_t* __restrict__ offsets, uint32_t T, uint32_t bid) {
    constexpr int R = 1 << RB;
    constexpr uint32_t kTileKeys = kBlock * ITEMS;
    __shared__ uint32_t s_cnt[4][R];
    __shared__ uint32_t s_goff[R];
    __shared__ uint32_t s_tdo[R];
    __shared__ uint32_t s_k[kTileKeys];
    __shared__ uint32_t s_v[kTileKeys];
    __shared__ uint32_t s_scan[4];
    const uint32_t n = min(*d_n, cap);
    const uint32_t tile = bid;
    const uint32_t base = tile * kTileKeys;
    if (base >= n) return;
    for (int i = threadIdx.x; i < 4 * R; i += kBlock) (&s_cnt[0][0])[i] = 0u;
    __syncthreads();

    const int w = wave_id(), l = lane_id();
    const uint32_t wbase = base + (uint32_t)w * (ITEMS * 64);
    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t pos = wbase + k * 64 + l;
        const bool ok = pos < n;
        key[k] = ok ? kin[pos] : 0u;
        val[k] = ok ? vin[pos] : 0u;
    }
    // stable rank inside the wave: lanes with the same digit found by
    // RB ballots; items processed in tile order
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t pos = wbase + k * 64 + l;
        const bool ok = pos < n;
        const uint32_t d = (key[k] >> shift) & (R - 1);
        uint64_t m = __ballot(ok);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const uint32_t below = (uint32_t)__popcll(m & lt);
        const uint32_t cnt = (uint32_t)__popcll(m);
        const uint32_t cur = ok ? s_cnt[w][d] : 0u;
        rank[k] = cur + below;
        if (ok && l == __ffsll((long long)m) - 1) s_cnt[w][d] = cur + cnt;
    }
    __syncthreads();
    // the digit's count in the tiles before this one, and in all
    uint32_t before = 0, all = 0;
    if (threadIdx.x < R) {
        if (FOLD) {
            const uint32_t tiles = (n + kTileKeys - 1u) / kTileKeys;
            for (uint32_t t0 = 0; t0 < tiles; t0 += 16u) {
                uint32_t c[16];
#pragma unroll
                for (uint32_t u = 0; u < 16u; ++u)
                    c[u] = t0 + u < tiles ? offsets[(size_t)(t0 + u) * R + threadIdx.x] : 0u;
#pragma unroll
                for (uint32_t u = 0; u < 16u; ++u) {
                    before += t0 + u < tile ? c[u] : 0u;
                    all += c[u];
                }
            }
        } else {
            before = offsets[(size_t)threadIdx.x * T + tile];
            all = totals[threadIdx.x];
        }
    }
    uint32_t total = 0;
    if (threadIdx.x < R) {
        const int d = threadIdx.x;
        const uint32_t c0 = s_cnt[0][d], c1 = s_cnt[1][d], c2 = s_cnt[2][d], c3 = s_cnt[3][d];
        s_cnt[0][d] = 0u;
        s_cnt[1][d] = c0;
        s_cnt[2][d] = c0 + c1;
        s_cnt[3][d] = c0 + c1 + c2;
        total = c0 + c1 + c2 + c3;
    }
    uint32_t tsum;
    const uint32_t tdo = block_excl_scan<kBlock / 64>(total, &tsum, s_scan);
    // digit bases: exclusive scan of the digit totals
    const uint32_t dbase = block_excl_scan<kBlock / 64>(all, &tsum, s_scan);
    if (threadIdx.x < R) {
        s_tdo[threadIdx.x] = tdo;
        s_goff[threadIdx.x] = dbase + before - tdo;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t pos = wbase + k * 64 + l;
        if (pos < n) {
            const uint32_t d = (key[k] >> shift) & (R - 1);
            const uint32_t lp = s_tdo[d] + s_cnt[w][d] + rank[k];
            s_k[lp] = key[k];
            s_v[lp] = val[k];
        }
    }
    __syncthreads();
    const uint32_t cnt_tile = min(kTileKeys, n - base);
    for (uint32_t j = threadIdx.x; j < cnt_tile; j += kBlock) {
        const uint32_t k = s_k[j];
        const uint32_t g = s_goff[(k >> shift) & (R - 1)] + j;
        kout[g] = k;
        vout[g] = s_v[j];
    }
}

template <int RB, int ITEMS, bool FOLD>
__global__ __launch_bounds__(kBlock) void k_sort_down(const uint32_t* __restrict__ kin,
                                                      const uint32_t* __restrict__ vin,
                                                      uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                      const uint32_t* d_n, uint32_t cap, int shift,
                                                      const uint32_t* __restrict__ totals,
                                                      const uint32_t* __restrict__ offsets, uint32_t T) {
    sort_down_body<RB, ITEMS, FOLD>(kin, vin, kout, vout, d_n, cap, shift, totals, offsets, T, blockIdx.x);
}

// pass `pass` of the sorts of many grids (UniJob): scratch layout as
// sort_impl (per-pass digit totals, then the counts matrix)
template <int RB>
__global__ __launch_bounds__(kBlock) void k_multi_sort_up(const UniJob* __restrict__ jobs,
                                                          const MultiEntry* __restrict__ e, uint32_t ne, int pass) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    sort_up_body<RB, kSortItems, false>(j.k[pass & 1], &j.h->P1, j.cap_P, pass * RB, j.sort + (size_t)j.passes * (1 << RB), j.T, bid);
}

template <int RB>
__global__ __launch_bounds__(kBlock) void k_multi_sort_scan(const UniJob* __restrict__ jobs,
                                                            const MultiEntry* __restrict__ e, uint32_t ne, int pass) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    sort_scan_body<RB, kSortItems>(&j.h->P1, j.cap_P, j.sort + (size_t)pass * (1 << RB), j.sort + (size_t)j.passes * (1 << RB),
                       j.T, bid);
}

template <int RB>
__global__ __launch_bounds__(kBlock) void k_multi_sort_down(const UniJob* __restrict__ jobs,
                                                            const MultiEntry* __restrict__ e, uint32_t ne, int pass) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const int i = pass & 1, o = i ^ 1;
    sort_down_body<RB, kSortItems, false>(j.k[i], j.v[i], j.k[o], j.v[o], &j.h->P1, j.cap_P, pass * RB,
                       j.sort + (size_t)pass * (1 << RB), j.sort + (size_t)j.passes * (1 << RB), j.T, bid);
}

template <int RB, int ITEMS, bool FOLD>
static void sort_impl(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, const uint32_t* d_n, uint32_t cap,
                      int key_bits, uint32_t* scratch, hipStream_t st) {
    constexpr int R = 1 << RB;
    const int passes = sort_passes(key_bits, RB);
    const uint32_t T = (uint32_t)sort_tiles(cap, ITEMS);
    if (T == 0) return;
    uint32_t* totals = scratch;
    uint32_t* counts = scratch + (size_t)passes * R;
    uint32_t *ki = k0, *vi = v0, *ko = k1, *vo = v1;
    const dim3 tiles(T), tb(kBlock);
    for (int p = 0; p < passes; ++p) {
        uint32_t* tot = totals + (size_t)p * R;
        hipLaunchKernelGGL((k_sort_up<RB, ITEMS, FOLD>), tiles, tb, 0, st, ki, d_n, cap, p * RB, counts, T);
        if (!FOLD) hipLaunchKernelGGL((k_sort_scan<RB, ITEMS>), dim3(R), tb, 0, st, d_n, cap, tot, counts, T);
        hipLaunchKernelGGL((k_sort_down<RB, ITEMS, FOLD>), tiles, tb, 0, st, ki, vi, ko, vo, d_n, cap, p * RB, tot,
                           counts, T);
        uint32_t* t = ki; ki = ko; ko = t;
        t = vi; vi = vo; vo = t;
    }
}

template <int RB>
static void sort_size(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, const uint32_t* d_n, uint32_t cap,
                      int key_bits, uint32_t* scratch, hipStream_t st) {
    if (sort_items(cap) == kSortItems) sort_impl<RB, kSortItems, false>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st);
    else if (sort_tiles(cap, kSmallItems) > kFoldTiles)
        sort_impl<RB, kSmallItems, false>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st);
    else
        sort_impl<RB, kSmallItems, true>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st);
}

uint32_t multi_sort_blocks(const UniJob& j, MultiSortStep step) {
    return step == MS_SCAN ? (1u << j.rb) : j.T;
}

template <int RB>
static void multi_sort_impl(MultiSortStep step, int pass, const UniJob* jobs, const MultiEntry* e, uint32_t ne,
                            uint32_t blocks, hipStream_t st) {
    const dim3 g(blocks), b(kBlock);
    if (step == MS_UP) hipLaunchKernelGGL(k_multi_sort_up<RB>, g, b, 0, st, jobs, e, ne, pass);
    else if (step == MS_SCAN) hipLaunchKernelGGL(k_multi_sort_scan<RB>, g, b, 0, st, jobs, e, ne, pass);
    else hipLaunchKernelGGL(k_multi_sort_down<RB>, g, b, 0, st, jobs, e, ne, pass);
}

void launch_multi_sort(MultiSortStep step, int rb, int pass, const UniJob* jobs, const MultiEntry* e, uint32_t ne,
                       uint32_t blocks, hipStream_t st) {
    if (ne == 0 || blocks == 0) return;
    switch (rb) {
        case 4: multi_sort_impl<4>(step, pass, jobs, e, ne, blocks, st); break;
        case 6: multi_sort_impl<6>(step, pass, jobs, e, ne, blocks, st); break;
        default: multi_sort_impl<8>(step, pass, jobs, e, ne, blocks, st); break;
    }
}

void launch_sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, const uint32_t* d_n, uint32_t cap,
                       int key_bits, int radix_bits, uint32_t* scratch, hipStream_t st) {
    switch (radix_bits) {
        case 4: sort_size<4>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st); break;
        case 6: sort_size<6>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st); break;
        default: sort_size<8>(k0, v0, k1, v1, d_n, cap, key_bits, scratch, st); break;
    }
}

// ------------------------------------------------------------------ scan
constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;   // 4096 values

size_t scan_scratch_bytes(uint32_t n) {
    const size_t tiles = ((size_t)n + kScanTile - 1) / kScanTile;
    return ((tiles + 4) * sizeof(uint32_t) + 15) & ~(size_t)15;
}

// one or two arrays of the same length, each with its own tile sums: grid row
// blockIdx.y takes one (two scans of half a million values: 31 us one after the
// other, 16 us side by side)
struct ScanArrays {
    const uint32_t* in[2];
    uint32_t* out[2];
    uint32_t* sums[2];
};

__global__ __launch_bounds__(kBlock) void k_scan_up(ScanArrays a, uint32_t n) {
    __shared__ uint32_t s_red[kBlock / 64];
    const uint32_t* __restrict__ in = a.in[blockIdx.y];
    uint32_t* __restrict__ sums = a.sums[blockIdx.y];
    const uint32_t base = blockIdx.x * kScanTile;
    uint32_t acc = 0;
    for (uint32_t i = base + threadIdx.x; i < min(n, base + (uint32_t)kScanTile); i += kBlock) acc += in[i];
    const uint32_t s = block_sum<kBlock / 64>(acc, s_red);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// exclusive scan of the tile sums in place (one block of 1024 threads)
__global__ __launch_bounds__(1024) void k_scan_sums(ScanArrays a, uint32_t tiles) {
    __shared__ uint32_t s_scan[16];
    uint32_t* sums = a.sums[blockIdx.y];
    uint32_t run = 0;
    for (uint32_t c0 = 0; c0 < tiles; c0 += 1024 * 4) {
        const uint32_t t0 = c0 + threadIdx.x * 4;
        uint32_t v[4], sum = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = t0 + k < tiles ? sums[t0 + k] : 0u;
            sum += v[k];
        }
        uint32_t tot;
        uint32_t pre = run + block_excl_scan<16>(sum, &tot, s_scan);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (t0 + k < tiles) sums[t0 + k] = pre;
            pre += v[k];
        }
        run += tot;
    }
}

__global__ __launch_bounds__(kBlock) void k_scan_down(ScanArrays a, uint32_t n, int inclusive) {
    __shared__ uint32_t s_scan[kBlock / 64];
    const uint32_t* __restrict__ in = a.in[blockIdx.y];
    uint32_t* __restrict__ out = a.out[blockIdx.y];
    const uint32_t* __restrict__ sums = a.sums[blockIdx.y];
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t sum = 0;
    if (base + kScanItems <= n) {
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4) {
            const uint4 q = *reinterpret_cast<const uint4*>(in + base + k);
            v[k] = q.x; v[k + 1] = q.y; v[k + 2] = q.z; v[k + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? in[base + k] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) sum += v[k];
    uint32_t agg;
    uint32_t run = sums[blockIdx.x] + block_excl_scan<kBlock / 64>(sum, &agg, s_scan);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t x = v[k];
        v[k] = inclusive ? run + x : run;
        run += x;
    }
    if (base + kScanItems <= n) {
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4)
            *reinterpret_cast<uint4*>(out + base + k) = make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (base + k < n) out[base + k] = v[k];
    }
}

static void scan_arrays(const ScanArrays& a, uint32_t count, uint32_t n, bool inclusive, hipStream_t st) {
    if (n == 0) return;
    const uint32_t tiles = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_up, dim3(tiles, count), dim3(kBlock), 0, st, a, n);
    hipLaunchKernelGGL(k_scan_sums, dim3(1, count), dim3(1024), 0, st, a, tiles);
    hipLaunchKernelGGL(k_scan_down, dim3(tiles, count), dim3(kBlock), 0, st, a, n, inclusive ? 1 : 0);
}

// in and out must be 16-byte aligned (device allocations are)
void launch_scan(const uint32_t* in, uint32_t* out, uint32_t n, bool inclusive, void* scratch, hipStream_t st) {
    scan_arrays(ScanArrays{{in, nullptr}, {out, nullptr}, {reinterpret_cast<uint32_t*>(scratch), nullptr}}, 1, n,
                inclusive, st);
}

void launch_scan_two(const uint32_t* const in[2], uint32_t* const out[2], uint32_t n, void* scratch, hipStream_t st) {
    char* p = reinterpret_cast<char*>(scratch);
    scan_arrays(ScanArrays{{in[0], in[1]}, {out[0], out[1]},
                           {reinterpret_cast<uint32_t*>(p), reinterpret_cast<uint32_t*>(p + scan_scratch_bytes(n))}},
                2, n, false, st);
}

}  // namespace sg
