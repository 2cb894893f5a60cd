// sg_build.hip -- grid construction kernels for gfx950.
//
// The build is device-resident: bounds, resolution, counts and totals live in
// the GridHeader in HBM, every kernel sizes itself from it, and no phase
// reads anything back to the host.  Counting, scanning and emission of each
// level are reduce-then-scan (a count kernel leaves one sum per tile; the
// emit kernel folds the sums of the tiles before it and rescans its own), so
// every pair lands at the slot that a serial scan of the counts in canonical
// order would give it: triangles (or sorted top pairs) ascending, then the
// reference's z/y/x loop order.
#include <cstddef>
#include <type_traits>

#include "sg_device.hpp"
#include "sg_kernels.hpp"

namespace sg {

// Triangles per thread in the top-level count and emission: four (16-byte
// loads), or one for scenes too small to give every CU a block that way, whose
// time is the longest lane's emission.
// (k_top_emit with one: 10,000-triangle soup 17.2 -> 6.8 us.  Two-level
// rebuilds with one / four, in us: soups of 300,000 triangles 98 / 103, 524,288
// 129 / 132, 600,000 140 / 140, 1,000,000 206 / 200; height fields of 520,000
// 126 / 131, 1,030,000 180 / 178, 2,093,058 359 / 328.  Uniform soups: 300,000
// 105 / 112, 600,000 161 / 164, 1,000,000 281 / 291.)
constexpr int kItems = 4;
constexpr uint32_t kSmallTop = 1u << 19;       // triangles up to which a thread takes one
constexpr uint32_t kStage = 1024;              // top pairs a tile stages in LDS, for each of a thread's triangles
static int top_items(uint32_t n) { return n <= kSmallTop ? 1 : kItems; }
static size_t top_tiles(uint32_t n, int items) { return ((size_t)n + kBlock * items - 1) / (kBlock * items); }

// --------------------------------------------------------------- init
// Zero the cell ranges and leaves; reset the header.
// The kernels of the build are written as bodies that take their block
// index and block count (bid, nb): the kernels below call them with
// blockIdx.x and gridDim.x, the multi-grid kernels (k_multi_*) with a
// grid's share of one launch over many grids.
SG_D void init_body(GridHeader* h, uint32_t n_tris, const ZeroSegs& segs, uint32_t bid, uint32_t nb) {
    if (bid == 0 && threadIdx.x == 0) {
        for (int i = 0; i < 3; ++i) {
            h->bmin_key[i] = 0xFFFFFFFFu;
            h->bmax_key[i] = 0u;
        }
        h->n_tris = n_tris;
        h->C1 = h->P1 = h->P1_valid = h->C2 = h->P2 = h->P2_valid = 0;
        h->need_P1 = h->need_C2 = h->need_P2 = 0;
        h->status = 0;
        h->leaf_sort = 0;
        h->oversize = 0;
    }
    const size_t stride = (size_t)nb * blockDim.x;
    for (int s = 0; s < segs.count; ++s) {
        uint4* p = reinterpret_cast<uint4*>(segs.ptr[s]);
        const size_t n16 = segs.bytes[s] >> 4;
        for (size_t i = (size_t)bid * blockDim.x + threadIdx.x; i < n16; i += stride)
            p[i] = make_uint4(0, 0, 0, 0);
    }
}


// --------------------------------------------------------------- bounds
// Scene AABB (the host loop of FastTwoLevelGridBuilder.h:75-81) as a device
// reduction; exact because min/max never round.  Coalesced SoA loads, four
// consecutive triangles per lane (one 16-byte load per SoA array, as the top
// count and emission read them; the arrays are 16-byte aligned).  The
// per-triangle records (TriSoA::rec) are written when the vertices change
// (sg_scene_create / sg_scene_update, k_prep_tris), not here.  Each block
// leaves its six partial keys in `part`; k_params folds them (no
// same-address atomics).
SG_D void bounds_body(const TriSoA& t, uint32_t n, uint32_t* __restrict__ part, uint32_t bid, uint32_t nb) {
    __shared__ uint32_t s_red[6][kBlock / 64];
    uint32_t k[6] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u, 0u, 0u};
    for (uint32_t i0 = (bid * kBlock + threadIdx.x) * 4u; i0 < n; i0 += nb * kBlock * 4u) {
        if (i0 + 4u <= n) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float4 p = reinterpret_cast<const float4*>(t.v[a])[i0 / 4];
                const float4 q = reinterpret_cast<const float4*>(t.v[3 + a])[i0 / 4];
                const float4 r = reinterpret_cast<const float4*>(t.v[6 + a])[i0 / 4];
                const uint32_t m0 = min(min(fkey(p.x), fkey(p.y)), min(fkey(p.z), fkey(p.w)));
                const uint32_t m1 = min(min(fkey(q.x), fkey(q.y)), min(fkey(q.z), fkey(q.w)));
                const uint32_t m2 = min(min(fkey(r.x), fkey(r.y)), min(fkey(r.z), fkey(r.w)));
                const uint32_t x0 = max(max(fkey(p.x), fkey(p.y)), max(fkey(p.z), fkey(p.w)));
                const uint32_t x1 = max(max(fkey(q.x), fkey(q.y)), max(fkey(q.z), fkey(q.w)));
                const uint32_t x2 = max(max(fkey(r.x), fkey(r.y)), max(fkey(r.z), fkey(r.w)));
                k[a] = min(k[a], min(m0, min(m1, m2)));
                k[3 + a] = max(k[3 + a], max(x0, max(x1, x2)));
            }
        } else {
            for (uint32_t i = i0; i < n; ++i)
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const uint32_t k0 = fkey(t.v[a][i]), k1 = fkey(t.v[3 + a][i]), k2 = fkey(t.v[6 + a][i]);
                    k[a] = min(k[a], min(k0, min(k1, k2)));
                    k[3 + a] = max(k[3 + a], max(k0, max(k1, k2)));
                }
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            k[a] = min(k[a], (uint32_t)__shfl_xor(k[a], d, 64));
            k[3 + a] = max(k[3 + a], (uint32_t)__shfl_xor(k[3 + a], d, 64));
        }
    }
    if (lane_id() == 0)
        for (int a = 0; a < 6; ++a) s_red[a][wave_id()] = k[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        uint32_t r = s_red[a][0];
        for (int w = 1; w < kBlock / 64; ++w) r = a < 3 ? min(r, s_red[a][w]) : max(r, s_red[a][w]);
        part[6 * bid + a] = r;
    }
}

// The first launch of a build: the zeroing of the build's segments and the
// bounds reduction, which touch disjoint memory, share one launch (their
// writes and reads then overlap instead of following each other).  Blocks
// below nb_bounds also reduce the bounds; every block zeroes.
__global__ __launch_bounds__(kBlock) void k_init_bounds(GridHeader* h, uint32_t n_tris, ZeroSegs segs, TriSoA t,
                                                        uint32_t* __restrict__ part, uint32_t nb_bounds) {
    init_body(h, n_tris, segs, blockIdx.x, gridDim.x);
    if (blockIdx.x < nb_bounds) bounds_body(t, n_tris, part, blockIdx.x, nb_bounds);
}

// --------------------------------------------------------------- params
// thread 0 of k_params: the folded bounds keys, then (derive) resolution,
// cell sizes and status; s_crcp receives the traversal cell_rcp
SG_D void fold_params(GridHeader* h, const BuildArgs& a, const uint32_t (*s_red)[kBlock / 64], int derive,
                      float* s_crcp) {
    for (int i = 0; i < 6; ++i) {
        uint32_t r = s_red[i][0];
        for (int w = 1; w < kBlock / 64; ++w) r = i < 3 ? min(r, s_red[i][w]) : max(r, s_red[i][w]);
        if (i < 3) h->bmin_key[i] = r;
        else h->bmax_key[i - 3] = r;
    }
    if (!derive) return;
    float mn[3], mx[3], cs[3], rcp[3], crcp[3];
    int32_t res[3];
    for (int i = 0; i < 3; ++i) {
        mn[i] = fkey_inv(h->bmin_key[i]);
        mx[i] = fkey_inv(h->bmax_key[i]);
    }
    const bool ok = derive_params(mn, mx, h->n_tris, a.lambda, a.top_divisor, a.fixed_res, res, cs, rcp, crcp);
    const uint64_t C = ok ? (uint64_t)res[0] * (uint64_t)res[1] * (uint64_t)res[2] : 0;
    uint32_t bad = 0;
    if (!ok) bad |= ST_INVALID;
    else if (C >= (1ull << 24)) bad |= ST_TOO_MANY_CELLS;
    else if (C > a.cap_C1) bad |= ST_CAP_C1;
    for (int i = 0; i < 3; ++i) {
        h->bmin[i] = mn[i];
        h->bmax[i] = mx[i];
        h->res[i] = ok ? res[i] : 0;
        h->cs[i] = ok ? cs[i] : 0.f;
        h->rcp_build[i] = ok ? rcp[i] : 0.f;
        h->cell_rcp[i] = ok ? crcp[i] : 0.f;
        s_crcp[i] = h->cell_rcp[i];
    }
    h->C1 = bad ? 0u : (uint32_t)C;
    if (bad) h->status |= bad;
}

// the leaf cell size table
SG_D void leaf_sizes(GridHeader* h, const float* s_crcp) {
    for (uint32_t i = threadIdx.x; i < 3u * 256u; i += kBlock) {
        const uint32_t d = i >> 8, c = i & 255u;
        h->leaf_size[d][c] = 1.f / (s_crcp[d] * (float)c);
    }
}

// Resolution and cell sizes from the reduced bounds, once (one thread):
// GridBuilder::computeResolution (GridBuilder.h:41-62), the two-level top
// resolution (FastTwoLevelGridBuilder.h:87-102) and the cell sizes of
// FastSimpleGridBuilder.h:114-117 / SimpleGrid.h:99-107.  One block: first
// the bounds partials of the nb bounds blocks are folded into the header;
// with derive the block then fills the leaf cell size table.
SG_D void fold_partials(GridHeader* h, const BuildArgs& a, const uint32_t* __restrict__ part, uint32_t nb, int derive,
                        float* s_crcp) {
    __shared__ uint32_t s_red[6][kBlock / 64];
    uint32_t k[6] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u, 0u, 0u};
    // four partials per thread and step, loaded before any is folded (one
    // memory round trip per step, not per partial)
    for (uint32_t b0 = threadIdx.x; b0 < nb; b0 += 4u * kBlock) {
        uint32_t v[4][6];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t b = b0 + (uint32_t)u * kBlock;
#pragma unroll
            for (int i = 0; i < 6; ++i) v[u][i] = b < nb ? part[6 * b + i] : (i < 3 ? 0xFFFFFFFFu : 0u);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 6; ++i) k[i] = i < 3 ? min(k[i], v[u][i]) : max(k[i], v[u][i]);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        for (int i = 0; i < 6; ++i) {
            const uint32_t o = (uint32_t)__shfl_xor(k[i], d, 64);
            k[i] = i < 3 ? min(k[i], o) : max(k[i], o);
        }
    if (lane_id() == 0)
        for (int i = 0; i < 6; ++i) s_red[i][wave_id()] = k[i];
    __syncthreads();
    if (threadIdx.x == 0) fold_params(h, a, s_red, derive, s_crcp);
    __syncthreads();
}

SG_D void params_body(GridHeader* h, const BuildArgs& a, const uint32_t* __restrict__ part, uint32_t nb, int derive) {
    __shared__ float s_crcp[3];
    fold_partials(h, a, part, nb, derive, s_crcp);
    if (derive) leaf_sizes(h, s_crcp);
}


__global__ __launch_bounds__(kBlock) void k_params(GridHeader* h, BuildArgs a, const uint32_t* __restrict__ part,
                                                   uint32_t nb, int derive) {
    params_body(h, a, part, nb, derive);
}

// grid parameters as every emission lane needs them (uniform loads)
struct Params {
    v3 gmin, cs, rcp, resf;
    uint32_t rx, rxy;
    bool ok;
};

SG_D Params read_params(const GridHeader* h) {
    Params p;
    p.gmin = mk(h->bmin[0], h->bmin[1], h->bmin[2]);
    p.cs = mk(h->cs[0], h->cs[1], h->cs[2]);
    p.rcp = mk(h->rcp_build[0], h->rcp_build[1], h->rcp_build[2]);
    p.resf = mk((float)h->res[0], (float)h->res[1], (float)h->res[2]);
    p.rx = (uint32_t)h->res[0];
    p.rxy = f2u(p.resf.x * p.resf.y);
    p.ok = h->C1 != 0;
    return p;
}

// BBox::empty + extend x3, src/Primitive/BBox.hpp:78-82,109-119
SG_D void tri_bounds(v3 a, v3 b, v3 c, v3& mn, v3& mx) {
    mn = vmin(vmin(vmin(mk(3.402823466e+38f, 3.402823466e+38f, 3.402823466e+38f), a), b), c);
    mx = vmax(vmax(vmax(mk(-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f), a), b), c);
}

// countRefs cell range, src/Control/Algorithm/FastBuildKernels.h:47-69
SG_D uint32_t top_range(const Params& p, v3 mn, v3 mx, uint32_t lo[3], uint32_t hi[3]) {
    v3 lof = vmax(mk(0.f, 0.f, 0.f), (mn - p.gmin) * p.rcp + mk(-kEps, -kEps, -kEps));
    v3 hif = vmin(p.resf - mk(1.f, 1.f, 1.f), (mx - p.gmin) * p.rcp + mk(kEps, kEps, kEps));
    lo[0] = f2u(lof.x); lo[1] = f2u(lof.y); lo[2] = f2u(lof.z);
    hi[0] = f2u(hif.x); hi[1] = f2u(hif.y); hi[2] = f2u(hif.z);
    if (hi[0] < lo[0] || hi[1] < lo[1] || hi[2] < lo[2]) return 0u;
    return (hi[0] - lo[0] + 1u) * (hi[1] - lo[1] + 1u) * (hi[2] - lo[2] + 1u);
}

// buildUnsortedGrid's per-triangle emission, src/Control/Algorithm/FastBuildKernels.h:130-212
SG_D void top_emit_one(const Params& P, const v3& v0, const v3& v1, const v3& v2, uint32_t i, uint32_t slot,
                       uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
    v3 mn, mx;
    uint32_t lo[3], hi[3];
    tri_bounds(v0, v1, v2, mn, mx);
    top_range(P, mn, mx, lo, hi);
    if (hi[0] - lo[0] > 0u && hi[1] - lo[1] > 0u && hi[2] - lo[2] > 0u) {
        const uint32_t dummy = f2u(P.resf.x * P.resf.y * P.resf.z);
        const v3 n_ = normalize(cross(v1 - v0, v2 - v0));
        const v3 half = scl(P.cs, 0.5f);
        const v3 c0 = (mk((float)lo[0], (float)lo[1], (float)lo[2]) * P.cs + P.gmin) + half;
        v3 cc;
        cc.z = c0.z - P.cs.z;
        for (uint32_t z = lo[2]; z <= hi[2]; ++z) {
            cc.z += P.cs.z;
            cc.y = c0.y - P.cs.y;
            for (uint32_t y = lo[1]; y <= hi[1]; ++y) {
                cc.y += P.cs.y;
                cc.x = c0.x - P.cs.x;
                for (uint32_t x = lo[0]; x <= hi[0]; ++x, ++slot) {
                    cc.x += P.cs.x;
                    const v3 dv = scl(n_, dot(cc - v0, n_));
                    const bool acc = fabsf(dv.x) <= half.x + kEps && fabsf(dv.y) <= half.y + kEps &&
                                     fabsf(dv.z) <= half.z + kEps;
                    keys[slot] = acc ? x + y * P.rx + z * P.rxy : dummy;
                    vals[slot] = i;
                }
            }
        }
    } else {
        for (uint32_t z = lo[2]; z <= hi[2]; ++z)
            for (uint32_t y = lo[1]; y <= hi[1]; ++y)
                for (uint32_t x = lo[0]; x <= hi[0]; ++x, ++slot) {
                    keys[slot] = x + y * P.rx + z * P.rxy;
                    vals[slot] = i;
                }
    }
}

// ------------------------------------------------------ top level emission
// countRefs + InclusiveScan + buildUnsortedGrid of
// src/Control/Algorithm/FastBuildKernels.h:31-215 as reduce-then-scan: a
// count kernel leaves one sum per tile of 1024 or 256 triangles, the emit kernel folds
// the sums of the tiles before it, rescans its own counts and writes every
// triangle's pairs at its slot.  kItems consecutive triangles per lane (one
// 16-byte load per SoA array); the emit kernel keeps the lane's vertices in
// registers from the count to the emission (reloading them after the scans
// fetched the arrays 2.3 times: a wave of blocks touches more than an XCD's
// L2 holds).
template <int ITEMS>
SG_D void top_counts(const Params& P, const TriSoA& t, uint32_t n, uint32_t i0, uint32_t cnt[ITEMS],
                     float f[9][ITEMS]) {
    for (int j = 0; j < ITEMS; ++j) cnt[j] = 0;
    if (!P.ok || i0 >= n) return;
    if (ITEMS == 4 && i0 + 4 <= n) {
#pragma unroll
        for (int c = 0; c < 9; ++c) {
            const float4 q = reinterpret_cast<const float4*>(t.v[c])[i0 / 4];
            f[c][0] = q.x; f[c][1 % ITEMS] = q.y; f[c][2 % ITEMS] = q.z; f[c][3 % ITEMS] = q.w;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 9; ++c)
#pragma unroll
            for (int j = 0; j < ITEMS; ++j) f[c][j] = i0 + j < n ? t.v[c][i0 + j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        if (i0 + j < n) {
            v3 mn, mx;
            uint32_t lo[3], hi[3];
            tri_bounds(mk(f[0][j], f[1][j], f[2][j]), mk(f[3][j], f[4][j], f[5][j]), mk(f[6][j], f[7][j], f[8][j]),
                       mn, mx);
            cnt[j] = top_range(P, mn, mx, lo, hi);
        }
    }
}

template <int ITEMS>
SG_D void top_count_body(const TriSoA& t, uint32_t n, const GridHeader* h, uint32_t* __restrict__ sums,
                         uint32_t* __restrict__ dbg_counts, uint32_t bid) {
    __shared__ uint32_t s_red[kBlock / 64];
    const Params P = read_params(h);
    const uint32_t i0 = bid * (kBlock * ITEMS) + threadIdx.x * ITEMS;
    uint32_t cnt[ITEMS];
    float f[9][ITEMS];
    top_counts<ITEMS>(P, t, n, i0, cnt, f);
    if (dbg_counts)
        for (int j = 0; j < ITEMS; ++j)
            if (i0 + j < n) dbg_counts[i0 + j] = cnt[j];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) sum += cnt[j];
    const uint32_t s = block_sum<kBlock / 64>(sum, s_red);
    if (threadIdx.x == 0) sums[bid] = s;
}

template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_top_count(TriSoA t, uint32_t n, GridHeader* h,
                                                      uint32_t* __restrict__ sums,
                                                      uint32_t* __restrict__ dbg_counts) {
    top_count_body<ITEMS>(t, n, h, sums, dbg_counts, blockIdx.x);
}

// The count of a small scene (one triangle per thread) also takes the place of
// k_params: every block folds the few bounds partials (at most 512) and derives
// the parameters for itself, block 0 leaves them in the header.  One launch of
// 3 us less (10,000 triangles: rebuild 37.9 -> 36.3 us).
__global__ __launch_bounds__(kBlock) void k_top_count_params(TriSoA t, uint32_t n, GridHeader* h, BuildArgs a,
                                                             const uint32_t* __restrict__ part, uint32_t nb,
                                                             uint32_t* __restrict__ sums,
                                                             uint32_t* __restrict__ dbg_counts) {
    __shared__ GridHeader s_h;   // its parameters only
    __shared__ float s_crcp[3];
    constexpr uint32_t kParamWords = offsetof(GridHeader, n_tris) / 4;   // bounds to cell_rcp
    if (threadIdx.x == 0) {
        s_h.n_tris = n;
        s_h.status = 0;
    }
    fold_partials(&s_h, a, part, nb, 1, s_crcp);
    if (blockIdx.x == 0) {
        if (threadIdx.x < kParamWords)
            reinterpret_cast<uint32_t*>(h)[threadIdx.x] = reinterpret_cast<const uint32_t*>(&s_h)[threadIdx.x];
        if (threadIdx.x == kParamWords) {
            h->C1 = s_h.C1;
            if (s_h.status) h->status |= s_h.status;
        }
        leaf_sizes(h, s_crcp);
    }
    top_count_body<1>(t, n, &s_h, sums, dbg_counts, blockIdx.x);
}

template <int ITEMS>
SG_D void top_emit_body(const TriSoA& t, uint32_t n, GridHeader* h, const BuildArgs& a, uint32_t* __restrict__ keys,
                        uint32_t* __restrict__ vals, const uint32_t* __restrict__ sums, uint32_t bid, uint32_t nb) {
    __shared__ uint32_t s_scan[kBlock / 64];
    __shared__ uint32_t s_k[(kStage * ITEMS)], s_v[(kStage * ITEMS)];
    const Params P = read_params(h);
    const uint32_t prefix = block_prefix_of<kBlock / 64>(sums, bid, s_scan);
    const uint32_t i0 = bid * (kBlock * ITEMS) + threadIdx.x * ITEMS;
    uint32_t cnt[ITEMS];
    float f[9][ITEMS];
    top_counts<ITEMS>(P, t, n, i0, cnt, f);
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) sum += cnt[j];
    uint32_t agg;
    const uint32_t local = block_excl_scan<kBlock / 64>(sum, &agg, s_scan);
    if (bid == nb - 1 && threadIdx.x == 0) {
        const uint32_t P1 = prefix + agg;
        h->need_P1 = P1;
        h->P1 = P1 <= a.cap_P1 ? P1 : a.cap_P1;
        if (P1 > a.cap_P1) atomicOr(&h->status, ST_CAP_P1);
    }
    if ((uint64_t)prefix + agg > a.cap_P1) return;   // flagged by the last tile
    if (agg <= (kStage * ITEMS)) {
        // the tile's pairs are one contiguous run: build it in LDS, then
        // write it out with full cache lines
        uint32_t ls = local;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (cnt[j])
                top_emit_one(P, mk(f[0][j], f[1][j], f[2][j]), mk(f[3][j], f[4][j], f[5][j]),
                             mk(f[6][j], f[7][j], f[8][j]), i0 + j, ls, s_k, s_v);
            ls += cnt[j];
        }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < agg; j += kBlock) {
            keys[prefix + j] = s_k[j];
            vals[prefix + j] = s_v[j];
        }
        return;
    }
    uint32_t slot = prefix + local;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        if (cnt[j])
            top_emit_one(P, mk(f[0][j], f[1][j], f[2][j]), mk(f[3][j], f[4][j], f[5][j]),
                         mk(f[6][j], f[7][j], f[8][j]), i0 + j, slot, keys, vals);
        slot += cnt[j];
    }
}

template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_top_emit(TriSoA t, uint32_t n, GridHeader* h, BuildArgs a,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals,
                                                     const uint32_t* __restrict__ sums) {
    top_emit_body<ITEMS>(t, n, h, a, keys, vals, sums, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------- ranges
// prepareCellRanges / prepareLeafCellRanges
// (src/Control/Algorithm/FastBuildKernels.h:218-313,
// src/Control/Algorithm/TwoLevelBuildKernels.h:458-536): a neighbour compare
// on the sorted keys writes {first, last+1} of every key below C; the dummy
// key's range is not stored.  Also records P_valid = index of the first
// dummy key.  Cells were zeroed by the build's first launch.
SG_D void ranges_body(const uint32_t* __restrict__ keys, const uint32_t* d_n, uint32_t cap, const uint32_t* d_C,
                      uint32_t* __restrict__ cells, uint32_t* d_pvalid, uint32_t bid, uint32_t nb) {
    const uint32_t n = min(*d_n, cap);
    const uint32_t C = *d_C;
    if (n == 0) {
        if (bid == 0 && threadIdx.x == 0) *d_pvalid = 0;
        return;
    }
    for (uint32_t i = bid * kBlock + threadIdx.x; i < n; i += nb * kBlock) {
        const uint32_t key = keys[i];
        const uint32_t prev = i > 0 ? keys[i - 1] : 0xFFFFFFFFu;
        const uint32_t next = i + 1 < n ? keys[i + 1] : 0xFFFFFFFFu;
        if (key < C) {
            if (key != prev) cells[2 * (size_t)key] = i;
            if (key != next) cells[2 * (size_t)key + 1] = i + 1;
            if (i + 1 == n) *d_pvalid = n;
        } else if (i == 0 || prev < C) {
            *d_pvalid = i;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_ranges(const uint32_t* __restrict__ keys, const uint32_t* d_n,
                                                   uint32_t cap, const uint32_t* d_C,
                                                   uint32_t* __restrict__ cells, uint32_t* d_pvalid) {
    ranges_body(keys, d_n, cap, d_C, cells, d_pvalid, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------ leaf cells
// countLeafLevelCells<false> + ExclusiveScan + prepareTopLevelCellRanges
// (src/Control/Algorithm/TwoLevelBuildKernels.h:40-127,
// src/Control/Algorithm/FastTwoLevelGridBuilder.h:256-294): count kernel +
// write kernel over tiles of 256 top cells.
SG_D uint32_t leaf_cell(const GridHeader* h, const BuildArgs& a, const uint32_t* __restrict__ ranges, uint32_t k,
                        uint32_t* bits) {
    const v3 cs = mk(h->cs[0], h->cs[1], h->cs[2]);
    const uint2 rg = reinterpret_cast<const uint2*>(ranges)[k];
    const uint32_t r = rg.y - rg.x;
    uint32_t rx = 1, ry = 1, rz = 1;
    if (r > a.leaf_min_refs) {
        const float vol = cs.x * cs.y * cs.z;
        const float m = cbrtpow(a.lambda_leaf * (float)r / vol);
        const v3 rf = scl(cs, m);
        rx = f2u(rf.x); ry = f2u(rf.y); rz = f2u(rf.z);
    }
    *bits = (r == 0 ? 0u : kNotEmpty) | (rx & 0xFFu) | ((ry & 0xFFu) << 8) | ((rz & 0xFFu) << 16);
    return rx * ry * rz;   // unmasked, as TwoLevelBuildKernels.h:81
}

// every leaf resolution in [1,255] (the packed bytes hold the whole value)
SG_D bool leaf_res_ok(uint32_t bits, uint32_t cnt) {
    const uint32_t rx = bits & 0xFFu, ry = (bits >> 8) & 0xFFu, rz = (bits >> 16) & 0xFFu;
    return rx >= 1 && ry >= 1 && rz >= 1 && rx * ry * rz == cnt;
}

__global__ __launch_bounds__(kBlock) void k_leaf_cells_count(GridHeader* h, BuildArgs a,
                                                             const uint32_t* __restrict__ ranges,
                                                             uint32_t* __restrict__ sums,
                                                             uint32_t* __restrict__ dbg_counts) {
    __shared__ uint32_t s_red[kBlock / 64];
    const uint32_t C1 = h->C1;
    const uint32_t base = blockIdx.x * kBlock;
    if (base >= C1) return;
    const uint32_t k = base + threadIdx.x;
    uint32_t cnt = 0, bits = 0;
    if (k < C1) {
        cnt = leaf_cell(h, a, ranges, k, &bits);
        if (!leaf_res_ok(bits, cnt)) atomicOr(&h->status, ST_LEAF_RES);
        if (dbg_counts) dbg_counts[k] = cnt;
    }
    const uint32_t s = block_sum<kBlock / 64>(cnt, s_red);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// empty leaf ranges, by the whole launch
SG_D void clear_leaves(uint32_t* __restrict__ leaves, uint32_t n) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x)
        reinterpret_cast<uint2*>(leaves)[k] = make_uint2(0u, 0u);
}

__global__ __launch_bounds__(kBlock) void k_leaf_cells_write(GridHeader* h, BuildArgs a,
                                                             const uint32_t* __restrict__ ranges,
                                                             uint32_t* __restrict__ cells,
                                                             const uint32_t* __restrict__ sums,
                                                         uint32_t* __restrict__ leaves) {
    __shared__ uint32_t s_scan[kBlock / 64];
    const uint32_t C1 = h->C1, failed = h->status & ~ST_NEG_EXTENT;
    const uint32_t base = blockIdx.x * kBlock;
    // A top cell reserves its leaf cells by the whole resolutions, its tile
    // writes those within the packed bytes: beyond 255 on an axis (flagged by
    // k_leaf_cells_count) the others are nobody's, so all are cleared here; so
    // are those of a build that has failed already.
    if (leaves && failed) clear_leaves(leaves, a.cap_C2);
    if (base >= C1) return;
    const uint32_t prefix = block_prefix_of<kBlock / 64>(sums, blockIdx.x, s_scan);
    const uint32_t k = base + threadIdx.x;
    uint32_t cnt = 0, bits = 0;
    if (k < C1) cnt = leaf_cell(h, a, ranges, k, &bits);
    uint32_t agg;
    const uint32_t local = block_excl_scan<kBlock / 64>(cnt, &agg, s_scan);
    if (k < C1) {
        reinterpret_cast<uint2*>(cells)[k] = make_uint2(prefix + local, bits);
        // an empty top cell's one leaf cell; the others' are written by the
        // tiles that emit their pairs, so nothing else clears them while the
        // leaf resolutions lie in 1..255 (then all are cleared above)
        if (leaves && !(bits & kNotEmpty) && prefix + local < a.cap_C2)
            reinterpret_cast<uint2*>(leaves)[prefix + local] = make_uint2(0u, 0u);
    }
    if (base + kBlock >= C1 && threadIdx.x == 0) {
        const uint32_t C2 = prefix + agg;
        h->need_C2 = C2;
        if (C2 > a.cap_C2) {
            atomicOr(&h->status, ST_CAP_C2);
            h->C2 = a.cap_C2;
        } else {
            h->C2 = C2;
        }
    }
}

// ------------------------------------------------------------- leaf pairs
// countLeafLevelRefs + InclusiveScan + writeLeafLevelRefs and the leaf-level
// radix sort (src/Control/Algorithm/TwoLevelBuildKernels.h:129-455,
// src/Control/Algorithm/FastTwoLevelGridBuilder.h:487-488,711-712).
//
// The leaf pairs of top cell k carry keys in [cells[k].x, cells[k].x + leaf
// cells of k), a range no other top cell uses, and pairs the plane test
// rejects carry the key C2.  The stable sort of all leaf pairs by key is
// therefore the concatenation, over top cells in order, of the stable sort of
// each top cell's accepted pairs, followed by every rejected pair in emission
// order.  Leaf tiles hold whole top cells: tile t covers the sorted top pairs
// from the first top-cell start at or after t*kLeafTile to the first one at
// or after (t+1)*kLeafTile.  The count kernel runs the plane test and leaves
// the tile's accepted and rejected totals, and for each pair where its box
// begins and which cells of it were accepted (PairBox); the emit kernel
// counts the tile's pairs per leaf cell in LDS, scans the counts, puts each
// pair's index into its cells' lists and writes accepted pairs to their final
// slots and rejected ones to the tail.  An oversize tile is emitted and sorted
// by one block; in a grid whose build has met one, its pairs are written in
// emission order by many, and GridHeader::leaf_sort enables a global stable
// radix sort of the accepted pairs (a no-op otherwise).
constexpr uint32_t kLeafTile = 512;                   // nominal sorted top pairs per leaf tile
constexpr int kLeafBlock = 512;                       // threads of the leaf emission kernel
constexpr int kBigBlock = 1024;                       // threads of its form for larger tiles
// What a tile may hold: accepted pairs, leaf cells, top pairs.  A tile beyond
// LeafSmall goes to the larger kernel, one beyond LeafBig is oversize.  The
// small kernel takes a tile's leaf cells in windows and a window's pairs in
// chunks of what its LDS holds (see leaf_emit_small).
struct LeafSmall {
    static constexpr uint32_t pairs = 4 * 4096, span = 65536, tops = 1536;
    static constexpr uint32_t chunk = 4096, window = 8192;
};
struct LeafBig {
    static constexpr uint32_t pairs = 65024, span = 16384, tops = 8192;
};
// A tile of the larger kernel is taken by several blocks: slice s holds the
// leaf cells whose lists begin in [s * kLeafSlice, (s+1) * kLeafSlice) of the
// tile's accepted pairs.  Every block counts the whole tile, then lists, sorts
// and writes its slice only.  Few tiles are so large, so their slices are small
// to use the chip, but each costs a count of the tile.  Rebuilds with slices of
// 2048 / 1024 / 512 pairs, in us: the 200,000-triangle sphere 150 / 143 / 142,
// with a leaf density of 4 172 / 167 / 198, with a top divisor of 12 168 / 162 /
// 190; the ruins scene 252 / 240 / 234; a 520,000-triangle height field with a
// leaf density of 16 230 / 243 / 257; eleven others within 2 %.
constexpr uint32_t kLeafSlice = 1024;
constexpr uint32_t kSliceShift = 24, kSlicesMax = (LeafBig::pairs + kLeafSlice - 1) / kLeafSlice;
constexpr int kTopBits = 13;                          // a list entry's top pair bits
static_assert(LeafBig::tops <= 1u << kTopBits && LeafBig::pairs < 65536u, "list entries and 16-bit counts");
static_assert(kSlicesMax <= 256u, "slice bits of a work item");

struct LeafParams {
    v3 gmin, cs;
    uint32_t rx, rxy, C1, C2, n_tris;
};

struct LeafSetup {
    v3 v0, v1, v2, org, cres;
    int lo[3], hp[3];
    uint32_t px;
};

SG_D LeafParams read_leaf_params(const GridHeader* h) {
    LeafParams L;
    L.gmin = mk(h->bmin[0], h->bmin[1], h->bmin[2]);
    L.cs = mk(h->cs[0], h->cs[1], h->cs[2]);
    L.rx = (uint32_t)h->res[0];
    L.rxy = (uint32_t)h->res[0] * (uint32_t)h->res[1];
    L.C1 = h->C1;
    L.C2 = h->C2;
    L.n_tris = h->n_tris;
    return L;
}

// leaf-cell box of one (top cell, triangle) pair; returns the number of leaf
// cells it spans, -1 for a negative extent
SG_D int leaf_range(const TriSoA& t, uint32_t key, uint32_t tri, const uint32_t* __restrict__ cells,
                    const LeafParams& L, LeafSetup& s) {
    const uint32_t tx = key % L.rx;
    const uint32_t ty = (key % L.rxy) / L.rx;
    const uint32_t tz = key / L.rxy;
    v3 mn, mx;
    load_tri_record(t.rec, tri, s.v0, s.v1, s.v2);
    tri_bounds(s.v0, s.v1, s.v2, mn, mx);
    const uint2 cell = reinterpret_cast<const uint2*>(cells)[key];
    s.px = cell.x;
    s.cres = mk((float)(cell.y & 0xFFu), (float)((cell.y >> 8) & 0xFFu), (float)((cell.y >> 16) & 0xFFu));
    s.org = mk((float)tx * L.cs.x + L.gmin.x, (float)ty * L.cs.y + L.gmin.y, (float)tz * L.cs.z + L.gmin.z);
    const v3 srcp = s.cres / L.cs;
    const v3 lof = (mn - s.org) * srcp + mk(-0.001f, -0.001f, -0.001f);
    const v3 hif = (mx - s.org) * srcp + mk(1.001f, 1.001f, 1.001f);
    int q;
    q = f2i(lof.x); s.lo[0] = q > 0 ? q : 0;
    q = f2i(lof.y); s.lo[1] = q > 0 ? q : 0;
    q = f2i(lof.z); s.lo[2] = q > 0 ? q : 0;
    int rc;
    rc = (int)s.cres.x; q = f2i(hif.x); s.hp[0] = rc < q ? rc : q;
    rc = (int)s.cres.y; q = f2i(hif.y); s.hp[1] = rc < q ? rc : q;
    rc = (int)s.cres.z; q = f2i(hif.z); s.hp[2] = rc < q ? rc : q;
    const int ex = s.hp[0] - s.lo[0], ey = s.hp[1] - s.lo[1], ez = s.hp[2] - s.lo[2];
    if (ex < 0 || ey < 0 || ez < 0) return -1;
    return ex * ey * ez;
}

// Visit the leaf cells of a pair in the reference's z/y/x order:
// f(key, accepted).  A triangle spanning more than one leaf cell on every axis
// keeps a cell only if the cell centre lies within half a cell (+EPS) of the
// triangle's plane on every axis.  Keys at or beyond C2 (a leaf level that
// overflowed its capacity) count as rejected.
template <class F>
SG_D void leaf_visit(const LeafParams& L, const LeafSetup& s, F&& f) {
    const uint32_t crx = f2u(s.cres.x), crxy = f2u(s.cres.x * s.cres.y);
    if (s.hp[0] - s.lo[0] > 1 && s.hp[1] - s.lo[1] > 1 && s.hp[2] - s.lo[2] > 1) {
        const v3 n_ = normalize(cross(s.v1 - s.v0, s.v2 - s.v0));
        const v3 scs = L.cs / s.cres;
        const v3 c0 = (mk((float)s.lo[0], (float)s.lo[1], (float)s.lo[2]) * scs + s.org) + scl(scs, 0.5f);
        v3 cc;
        cc.z = c0.z - scs.z;
        for (int z = s.lo[2]; z < s.hp[2]; ++z) {
            cc.z += scs.z;
            cc.y = c0.y - scs.y;
            for (int y = s.lo[1]; y < s.hp[1]; ++y) {
                cc.y += scs.y;
                cc.x = c0.x - scs.x;
                for (int x = s.lo[0]; x < s.hp[0]; ++x) {
                    cc.x += scs.x;
                    const v3 dv = scl(n_, dot(cc - s.v0, n_));
                    const bool acc = fabsf(dv.x) <= scs.x * 0.5f + kEps && fabsf(dv.y) <= scs.y * 0.5f + kEps &&
                                     fabsf(dv.z) <= scs.z * 0.5f + kEps;
                    const uint32_t key = (uint32_t)x + (uint32_t)y * crx + (uint32_t)z * crxy + s.px;
                    f(key, acc && key < L.C2);
                }
            }
        }
    } else {
        for (int z = s.lo[2]; z < s.hp[2]; ++z)
            for (int y = s.lo[1]; y < s.hp[1]; ++y)
                for (int x = s.lo[0]; x < s.hp[0]; ++x) {
                    const uint32_t key = (uint32_t)x + (uint32_t)y * crx + (uint32_t)z * crxy + s.px;
                    f(key, key < L.C2);
                }
    }
}

// set-up of sorted top pair i; 0 pairs for a negative extent (flagged) or a
// top level that overflowed its buffers (never follow an id outside the
// scene or the grid)
SG_D uint32_t leaf_pair(const TriSoA& t, const LeafParams& L, GridHeader* h, uint32_t key, uint32_t tri,
                        const uint32_t* __restrict__ cells, LeafSetup& s) {
    if (tri >= L.n_tris || key >= L.C1) return 0;
    const int c = leaf_range(t, key, tri, cells, L, s);
    if (c < 0) {
        atomicOr(&h->status, ST_NEG_EXTENT);
        return 0;
    }
    return (uint32_t)c;
}

// Wide leaf boxes: one triangle that crosses a finely divided top cell (a
// large triangle through a dense cluster) spans up to 255^3 leaf cells, and
// one lane walking them sets the time of the whole launch (10,368 + 66,612
// cells in a 502,000-triangle cluster: k_leaf_count 5.6 ms, its emission
// 8.6 ms).  A box of at least kWideBox cells is therefore visited by its
// block, one (y, z) row of leaf cells per thread (k_leaf_count lists it and
// k_leaf_scan or k_leaf_wide counts it; k_leaf_emit_big emits it in place, with
// the parallel emission k_leaf_wide_emit).
// Along a row the plane distance never changes direction -- each binary32
// operation between the cell centre and the distance is monotone -- so a
// row's accepted cells are one interval, found by two binary searches.  The
// cell centres are the running sums of leaf_visit, formed once per axis in
// LDS.  The rebuild of that cluster went from 14.6 to 0.37 ms.  Below kWideBox
// cells the lanes of a wave walk their boxes side by side; a shared visit
// costs its block about as long as such a walk.
constexpr uint32_t kWideBox = 1024;
constexpr uint32_t kWideCap = 1024;   // wide boxes a build counts this way; the rest are walked by their lanes
constexpr int kAxisMax = 256;      // leaf cells along an axis (resolution bytes)

SG_D bool plane_tested(const LeafSetup& s) {
    return s.hp[0] - s.lo[0] > 1 && s.hp[1] - s.lo[1] > 1 && s.hp[2] - s.lo[2] > 1;
}

// Monotone needs finite terms: coordinates below 1e18 keep every product of
// the distance in range (a normal of zeros, infinities or NaN then rejects
// every cell or, all zero, accepts every cell, in the search as in the walk).
SG_D bool finite_box(const LeafParams& L, const LeafSetup& s) {
    auto ok = [](v3 a) { return fabsf(a.x) < 1e18f && fabsf(a.y) < 1e18f && fabsf(a.z) < 1e18f; };
    return ok(s.v0) && ok(s.v1) && ok(s.v2) && ok(s.org) && ok(s.org + L.cs);
}

SG_D bool wide_box(const LeafParams& L, const LeafSetup& s, uint32_t c) { return c >= kWideBox && finite_box(L, s); }

// Every thread of the block, or with WAVE of the wave, calls this with the same
// pair.  f(r, key0, xa, xb) once per round of rows: cells [xa, xb) of the
// thread's row r are accepted, key0 the key of the row's cell 0 (xa == xb
// without a row).
template <bool WAVE = false, class F>
SG_D void wide_visit(const LeafParams& L, const LeafSetup& s, float (*tab)[kAxisMax], F&& f) {
    const int ex = s.hp[0] - s.lo[0], ey = s.hp[1] - s.lo[1], ez = s.hp[2] - s.lo[2];
    const uint32_t crx = f2u(s.cres.x), crxy = f2u(s.cres.x * s.cres.y);
    const bool plane = plane_tested(s);
    const v3 n_ = normalize(cross(s.v1 - s.v0, s.v2 - s.v0));
    const v3 scs = L.cs / s.cres;
    const int tid = WAVE ? lane_id() : (int)threadIdx.x, threads = WAVE ? 64 : (int)blockDim.x;
    auto sync = [&]() {
        if (WAVE) __threadfence_block();
        else __syncthreads();
    };
    sync();   // tab is free again
    if (tid < 3) {
        const int a = tid;
        const v3 c0 = (mk((float)s.lo[0], (float)s.lo[1], (float)s.lo[2]) * scs + s.org) + scl(scs, 0.5f);
        const float step = comp(scs, a);
        float c = comp(c0, a) - step;
        const int m = a == 0 ? ex : (a == 1 ? ey : ez);
        for (int i = 0; i < m && i < kAxisMax; ++i) {
            c += step;
            tab[a][i] = c;
        }
    }
    sync();
    const float hx = scs.x * 0.5f + kEps, hy = scs.y * 0.5f + kEps, hz = scs.z * 0.5f + kEps;
    const int rows = ey * ez;
    for (int r0 = 0; r0 < rows; r0 += threads) {
        const int r = r0 + tid;
        const bool live = r < rows;
        int xa = 0, xb = 0;
        uint32_t key0 = 0;
        if (live) {
            const int z = r / ey, y = r - z * ey;
            key0 = (uint32_t)s.lo[0] + (uint32_t)(s.lo[1] + y) * crx + (uint32_t)(s.lo[2] + z) * crxy + s.px;
            xb = ex;
            if (plane) {
                const float dy = (tab[1][y] - s.v0.y) * n_.y, dz = (tab[2][z] - s.v0.z) * n_.z;
                auto dist = [&](int x) { return ((tab[0][x] - s.v0.x) * n_.x + dy) + dz; };
                auto in = [&](float d) {
                    return fabsf(n_.x * d) <= hx && fabsf(n_.y * d) <= hy && fabsf(n_.z * d) <= hz;
                };
                // cells before the interval lie on one side of the plane, those
                // after it on the other
                const bool up = n_.x >= 0.f;
                int lo = 0, hi = ex;   // first cell not before the interval
                while (lo < hi) {
                    const int m = (lo + hi) >> 1;
                    const float d = dist(m);
                    if (!in(d) && (d < 0.f) == up) lo = m + 1;
                    else hi = m;
                }
                xa = lo;
                hi = ex;               // first cell after it
                while (lo < hi) {
                    const int m = (lo + hi) >> 1;
                    if (in(dist(m))) lo = m + 1;
                    else hi = m;
                }
                xb = lo;
            }
            const int room = key0 < L.C2 ? (int)min(L.C2 - key0, (uint32_t)ex) : 0;   // keys at C2 are rejected
            xb = min(xb, room);
            xa = min(xa, xb);
        }
        f((uint32_t)r, key0, xa, xb);
    }
}

// accepted cells of a wide box (the block's sum, known to every thread)
template <int NW>
SG_D uint32_t wide_count(const LeafParams& L, const LeafSetup& s, float (*tab)[kAxisMax], uint32_t* s_red) {
    uint32_t acc = 0;
    wide_visit(L, s, tab, [&](uint32_t, uint32_t, int xa, int xb) { acc += (uint32_t)(xb - xa); });
    return block_sum<NW>(acc, s_red);
}

// The leaf pairs of a wide box: accepted ones from slot pa in z/y/x order,
// the `rej` rejected ones from slot pr (all alike: key C2).
template <int NW>
SG_D void wide_emit(const LeafParams& L, const LeafSetup& s, float (*tab)[kAxisMax], uint32_t* s_scan, uint32_t tri,
                    uint32_t pa, uint32_t pr, uint32_t rej, uint32_t cap, uint32_t* __restrict__ keys,
                    uint32_t* __restrict__ vals) {
    wide_visit(L, s, tab, [&](uint32_t, uint32_t key0, int xa, int xb) {
        uint32_t agg;
        uint32_t p = pa + block_excl_scan<NW>((uint32_t)(xb - xa), &agg, s_scan);
        for (int x = xa; x < xb; ++x, ++p)
            if (p < cap) {
                keys[p] = key0 + (uint32_t)x;
                vals[p] = tri;
            }
        pa += agg;
    });
    for (uint32_t j = threadIdx.x; j < rej; j += NW * 64)
        if (pr + j < cap) {
            keys[pr + j] = L.C2;
            vals[pr + j] = tri;
        }
}

// PairBox: what the emission needs of a top pair, so that it neither gathers
// the triangle nor forms its box and plane again.  x: the leaf cell of the
// box's corner within its top cell (16 bits) and the box's extents less one
// (5 bits each); y: the accepted cells, bit k for the k-th in z/y/x order.
// Boxes of up to 32 cells with a corner below 2^16 have this form.  Larger
// ones are stored in the pool of masks: x is kBoxOpen and the place of
// {corner, extents (8 bits each) and kBoxFull when every cell is accepted,
// otherwise the masks, 32 cells each}, y the number of accepted cells.  (406,002
// triangles, three large ones across each of 2,000 top cells: rebuild 568 us with
// such boxes visited again by the emission, 170 stored.)  Boxes that a block
// visits together, and those that find no place, are kBoxWide: the emission
// visits them again.  Pairs without leaf cells: empty.
constexpr uint32_t kBoxOpen = 0x80000000u, kBoxEmpty = 0x7FFFFFFFu, kBoxWide = 0xFFFFFFFFu;
constexpr uint32_t kBoxFull = 0x80000000u;
// The pool is cut in kPools parts, each with its counter in a cache line of its
// own, used by every kPools-th block: adds of many waves to one counter wait
// for each other.
constexpr uint32_t kPools = 16, kPoolStride = 16;

struct BoxPool {
    uint32_t* words;   // kPools parts of `part` words
    uint32_t part;
};

// the leaf cell of the box's corner within its top cell
SG_D uint32_t box_corner(const LeafSetup& s) {
    const uint32_t crx = f2u(s.cres.x), crxy = f2u(s.cres.x * s.cres.y);
    return (uint32_t)s.lo[0] + (uint32_t)s.lo[1] * crx + (uint32_t)s.lo[2] * crxy;
}

struct BoxExtent {
    uint32_t corner, ex, ey, ez;
};

SG_D BoxExtent box_extent(uint2 box, const uint32_t* __restrict__ pool) {
    BoxExtent e;
    if (box.x < kBoxOpen) {
        e.corner = box.x & 0xFFFFu;
        e.ex = ((box.x >> 16) & 31u) + 1u;
        e.ey = ((box.x >> 21) & 31u) + 1u;
        e.ez = ((box.x >> 26) & 31u) + 1u;
    } else {
        const uint32_t* q = pool + (box.x & ~kBoxOpen);
        const uint32_t x = q[1];
        e.corner = q[0];
        e.ex = x & 0xFFu;
        e.ey = (x >> 8) & 0xFFu;
        e.ez = (x >> 16) & 0xFFu;
    }
    return e;
}

// cells of a box of the first form (0: empty)
SG_D uint32_t box_cells(uint32_t x) {
    if (x >= kBoxEmpty) return 0u;
    return (((x >> 16) & 31u) + 1u) * (((x >> 21) & 31u) + 1u) * (((x >> 26) & 31u) + 1u);
}

// rejected cells of a box (not kBoxWide)
SG_D uint32_t box_rejects(uint2 box, const uint32_t* __restrict__ pool) {
    if (box.x == kBoxEmpty) return 0u;
    const BoxExtent e = box_extent(box, pool);
    return e.ex * e.ey * e.ez - (box.x < kBoxOpen ? (uint32_t)__popc(box.y) : box.y);
}

// the leaf cells [lo, hi] between the first and the last cell of a box
SG_D void box_bounds(const BoxExtent& e, uint32_t first, uint32_t crx, uint32_t cry, uint32_t& lo, uint32_t& hi) {
    lo = first + e.corner;
    hi = lo + e.ex - 1u + (e.ey - 1u + (e.ez - 1u) * cry) * crx;
}

// f(leaf cell) for every accepted cell of a box of the first form, `first` the
// tile's index of the top cell's leaf cell 0, crx and cry its resolution along
// x and y
template <class F>
SG_D void box_visit(uint2 box, uint32_t first, uint32_t crx, uint32_t cry, F&& f) {
    const uint32_t ex = ((box.x >> 16) & 31u) + 1u, ey = ((box.x >> 21) & 31u) + 1u;
    uint32_t row = first + (box.x & 0xFFFFu), y = 0, x = 0;
    const uint32_t next = (cry - (ey - 1u)) * crx;   // from a slice's last row to the next slice's first
    for (uint32_t m = box.y; m; m >>= 1) {
        if (m & 1u) f(row + x);
        if (++x == ex) {
            x = 0;
            const bool last = ++y == ey;
            row += last ? next : crx;
            y = last ? 0u : y;
        }
    }
}

// the same for a stored box: the plane accepts few of its cells, so its mask is
// read by its set bits (places below 2^10 divided exactly by a multiplication)
template <class F>
SG_D void stored_visit(uint2 box, const uint32_t* __restrict__ pool, uint32_t first, uint32_t crx, uint32_t cry,
                       F&& f) {
    if (box.y == 0u) return;
    const BoxExtent e = box_extent(box, pool);
    const uint32_t* q = pool + (box.x & ~kBoxOpen);
    const bool full = (q[1] & kBoxFull) != 0u;
    const uint32_t n = e.ex * e.ey * e.ez, crxy = crx * cry;
    const float rx = 1.f / (float)e.ex, ry = 1.f / (float)e.ey;
    for (uint32_t k0 = 0; k0 < n; k0 += 32u) {
        uint32_t m = full ? 0xFFFFFFFFu : q[2u + (k0 >> 5)];
        if (n - k0 < 32u) m &= (1u << (n - k0)) - 1u;
        for (; m; m &= m - 1u) {
            const uint32_t k = k0 + (uint32_t)__ffs((int)m) - 1u, r = (uint32_t)(((float)k + 0.5f) * rx),
                           z = (uint32_t)(((float)r + 0.5f) * ry);
            f(first + e.corner + (k - r * e.ex) + (r - z * e.ey) * crx + z * crxy);
        }
    }
}

// Leaf tile of a sorted top pair: tile t holds the top cells that start in
// [t*kLeafTile, (t+1)*kLeafTile), so pair i belongs to tile
// floor(start of its top cell / kLeafTile).  Per tile the count kernel
// records (zero-initialised words, combined with atomicMax):
//   info[4t+0] = ~first pair   info[4t+1] = end pair
//   info[4t+2] = ~first leaf key   info[4t+3] = last leaf key + 1
//   info[4T+t] = 1 when a pair of the tile has a stored box (kBoxOpen)
//   info[5T+t] = 1 when one has a kBoxWide box
// and its accepted / rejected leaf-pair totals in sums[t] / sums[Tp + t].
SG_HD uint32_t leaf_sums_stride(uint32_t T) { return (T + 15u) & ~15u; }

// The wave's boxes that are stored (need: their words in the pool), with the
// plane test counted on the way: acc and box of those lanes.  The whole wave
// calls this.  A box of kCoopBox cells or more is visited by the wave, a row of
// cells per lane (see wide_visit), its mask put together in LDS: a lane alone
// walks a cell in some 60 ns, and its wave waits.  (401,002 triangles, 1,000 boxes
// of some 1,000 cells: k_leaf_count 149 -> 20 us; 603,002 triangles, 3,000 of
// some 300: 103 -> 55.  From 128 cells on, the ruins rebuild took 295 us for 238,
// from 512 on the two scenes 2 and 9 % longer.)
constexpr uint32_t kCoopBox = 256;
SG_D void store_boxes(const TriSoA& t, const LeafParams& L, GridHeader* h, uint32_t key, uint32_t tri,
                      const uint32_t* __restrict__ cells, const BoxPool& pool, uint32_t* __restrict__ pool_n,
                      uint32_t need, float (*tab)[kAxisMax], uint32_t* s_mask, uint32_t& acc, uint2& box) {
    const uint32_t part = blockIdx.x % kPools, inc = wave_incl_scan(need), l = (uint32_t)lane_id();
    uint32_t place = 0;
    if (l == 63u) place = atomicAdd(&pool_n[part * kPoolStride], inc);
    place = (uint32_t)__shfl((int)place, 63, 64) + inc - need;
    const bool room = place + need <= pool.part;   // otherwise the box is only counted
    uint32_t* words = pool.words + (size_t)part * pool.part + place;
    auto head = [&](const LeafSetup& s, uint32_t* w, bool full) {
        w[0] = box_corner(s);
        w[1] = (uint32_t)(s.hp[0] - s.lo[0]) | (uint32_t)(s.hp[1] - s.lo[1]) << 8 |
               (uint32_t)(s.hp[2] - s.lo[2]) << 16 | (full ? kBoxFull : 0u);
    };
    bool mine = need != 0u;
    for (uint64_t m = __ballot(need >= 2u + kCoopBox / 32u); m; m &= m - 1ull) {
        const int o = __ffsll((long long)m) - 1;
        LeafSetup s;
        const uint32_t c = leaf_pair(t, L, h, (uint32_t)__builtin_amdgcn_readlane((int)key, o),
                                     (uint32_t)__builtin_amdgcn_readlane((int)tri, o), cells, s);
        if (!finite_box(L, s)) continue;   // walked below
        const uint32_t ex = (uint32_t)(s.hp[0] - s.lo[0]);
        uint32_t n = 0;
        if (l < kWideBox / 32u) s_mask[l] = 0;
        wide_visit<true>(L, s, tab, [&](uint32_t r, uint32_t, int xa, int xb) {
            n += (uint32_t)(xb - xa);
            for (uint32_t k = r * ex + (uint32_t)xa, e = r * ex + (uint32_t)xb; k < e;) {
                const uint32_t to = min(e, (k | 31u) + 1u), c2 = to - k;
                atomicOr(&s_mask[k >> 5], (c2 < 32u ? (1u << c2) - 1u : 0xFFFFFFFFu) << (k & 31u));
                k = to;
            }
        });
        __threadfence_block();
        n = wave_sum(n);
        if (__builtin_amdgcn_readlane((int)room, o)) {
            const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)place, o);
            uint32_t* w = pool.words + (size_t)part * pool.part + at;
            if (l < (c + 31u) / 32u) w[2u + l] = s_mask[l];
            if (l == 0u) head(s, w, false);
        }
        __threadfence_block();   // s_mask is free again
        if ((int)l == o) {
            acc = n;
            mine = false;
        }
    }
    if (mine) {
        LeafSetup s;
        leaf_pair(t, L, h, key, tri, cells, s);
        if (need > 2u) {   // with a plane test
            uint32_t bit = 0, mask = 0, *w = words + 2;
            leaf_visit(L, s, [&](uint32_t, bool ok) {
                acc += ok ? 1u : 0u;
                mask |= ok ? 1u << (bit & 31u) : 0u;
                if ((++bit & 31u) == 0u) {
                    if (room) *w = mask;
                    ++w;
                    mask = 0;
                }
            });
            if (room && (bit & 31u)) *w = mask;
        }
        if (room) head(s, words, need == 2u);
    }
    if (need && room) box = make_uint2(kBoxOpen | (part * pool.part + place), acc);
}

// One sorted top pair per lane: the lane with the most leaf cells to visit
// sets a wave's time, and with four consecutive pairs per lane (one 16-byte
// load per array) those lanes ran four set-ups and visits in a row --
// height-field rebuild 0.387 -> 0.364 ms, ruins 0.392 -> 0.315 ms with one.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_leaf_count(
    TriSoA t, GridHeader* h, const uint32_t* __restrict__ top_keys, const uint32_t* __restrict__ top_vals,
    const uint32_t* __restrict__ ranges, const uint32_t* __restrict__ cells, uint32_t* __restrict__ sums,
    uint32_t* __restrict__ info, uint32_t T, uint32_t* __restrict__ dbg_counts, uint2* __restrict__ boxes,
    BoxPool pool, uint32_t* __restrict__ pool_n, uint32_t* __restrict__ pacc, uint32_t* __restrict__ prej) {
    constexpr int kSlots = 4;
    __shared__ uint32_t s_acc[kSlots], s_rej[kSlots], s_open[kSlots][2], s_info[kSlots][4];
    __shared__ float s_tab[kBlock / 64][3][kAxisMax];
    __shared__ uint32_t s_mask[kBlock / 64][kWideBox / 32];
    const uint32_t P1v = h->P1_valid;
    const uint32_t base = blockIdx.x * kBlock;
    if (base >= P1v) return;
    if (threadIdx.x < kSlots) s_acc[threadIdx.x] = s_rej[threadIdx.x] = 0;
    if (threadIdx.x < 2 * kSlots) s_open[threadIdx.x >> 1][threadIdx.x & 1] = 0;
    if (threadIdx.x < 4 * kSlots) s_info[threadIdx.x >> 2][threadIdx.x & 3] = 0;
    const LeafParams L = read_leaf_params(h);
    const uint32_t Tp = leaf_sums_stride(T);
    const uint32_t i = base + threadIdx.x;
    const uint32_t key = i < P1v ? top_keys[i] : 0u;
    const uint32_t tri = i < P1v ? top_vals[i] : 0u;
    // the block's first pair may sit in a top cell that starts far earlier:
    // slot 0 is that pair's tile, slots 1.. the tiles from base on
    const uint32_t first_key = top_keys[base];
    const uint32_t tile0 = first_key < L.C1 ? reinterpret_cast<const uint2*>(ranges)[first_key].x / kLeafTile : 0u;
    const uint32_t tile1 = base / kLeafTile;
    __syncthreads();
    const bool live = i < P1v && key < L.C1;
    const uint2 rg = live ? reinterpret_cast<const uint2*>(ranges)[key] : make_uint2(0u, 0u);
    uint32_t c = 0, acc = 0, need = 0;
    uint2 box = make_uint2(kBoxEmpty, 0u);
    bool counted = true;
    if (live) {
        LeafSetup st;
        c = leaf_pair(t, L, h, key, tri, cells, st);
        if (dbg_counts) dbg_counts[i] = c;
        if (c) {
            // a box of one leaf cell on some axis has no plane test: every
            // cell is accepted unless its key reaches C2, and the largest
            // key is that of the far corner -- then the count is the volume
            const uint32_t crx = f2u(st.cres.x), crxy = f2u(st.cres.x * st.cres.y), corner = box_corner(st);
            const uint32_t kmax = (uint32_t)(st.hp[0] - 1) + (uint32_t)(st.hp[1] - 1) * crx +
                                  (uint32_t)(st.hp[2] - 1) * crxy + st.px;
            const bool plane = plane_tested(st) || kmax >= L.C2;
            box.x = corner | (uint32_t)(st.hp[0] - st.lo[0] - 1) << 16 | (uint32_t)(st.hp[1] - st.lo[1] - 1) << 21 |
                    (uint32_t)(st.hp[2] - st.lo[2] - 1) << 26;
            if (c > 32u || corner >= 65536u) {
                box.x = kBoxWide;
                if (c < kWideBox) {
                    // (a top cell of more than 2^16 leaf cells makes its tile oversize)
                    if (corner < 65536u) need = 2u + (plane ? (c + 31u) / 32u : 0u);
                } else if (finite_box(L, st) && (pacc || plane)) {
                    // listed: counted by blocks, and for its emission
                    const uint32_t w = atomicAdd(&sums[2 * (size_t)Tp + 2], 1u);
                    if (w < kWideCap) sums[2 * (size_t)Tp + 4 + w] = i;
                    counted = !plane || w >= kWideCap;
                }
            }
            if (!plane) {
                acc = c;
                box.y = c >= 32u ? 0xFFFFFFFFu : (1u << c) - 1u;
            } else if (counted && !need) {
                uint32_t bit = 0;
                leaf_visit(L, st, [&](uint32_t, bool ok) {
                    acc += ok ? 1u : 0u;
                    box.y |= ok && bit < 32u ? 1u << bit : 0u;
                    ++bit;
                });
            }
        }
    }
    if (__builtin_expect(__ballot(need != 0u) != 0ull, 0))
        store_boxes(t, L, h, key, tri, cells, pool, pool_n, need, s_tab[wave_id()], s_mask[wave_id()], acc, box);
    if (live) {
        const uint32_t tile = rg.x / kLeafTile;
        boxes[i] = box;
        if (box.x >= kBoxOpen && tile < T) {
            const uint32_t slot = tile == tile0 ? 0u : tile - tile1 + 1u, wide = box.x == kBoxWide ? 1u : 0u;
            if (slot < kSlots) s_open[slot][wide] = 1u;
            else info[(4 + wide) * (size_t)T + tile] = 1u;
        }
        if (counted && pacc) {   // per-pair totals for the parallel emission of oversize tiles
            pacc[i] = acc;
            prej[i] = c - acc;
        }
        if (tile < T) {
            if (counted && !pacc) {
                const uint32_t slot = tile == tile0 ? 0u : tile - tile1 + 1u;
                if (slot < kSlots) {
                    if (acc) atomicAdd(&s_acc[slot], acc);
                    if (c - acc) atomicAdd(&s_rej[slot], c - acc);
                } else {
                    atomicAdd(&sums[tile], acc);
                    atomicAdd(&sums[Tp + tile], c - acc);
                }
            }
            if (rg.x == i) {   // first pair of its top cell
                const uint2 cl = reinterpret_cast<const uint2*>(cells)[key];
                const uint32_t nl = (cl.y & 0xFFu) * ((cl.y >> 8) & 0xFFu) * ((cl.y >> 16) & 0xFFu);
                // folded in LDS: the top cells of a tile, up to 512 where they
                // hold few pairs each, would wait for the same four words in
                // memory (502,000-triangle cluster, 9,000 such cells: k_leaf_count
                // 103 -> 10 us)
                const uint32_t slot = tile == tile0 ? 0u : tile - tile1 + 1u;
                const uint32_t v[4] = {~i, rg.y, ~cl.x, cl.x + nl};
                if (slot < kSlots)
                    for (int k = 0; k < 4; ++k) atomicMax(&s_info[slot][k], v[k]);
                else
                    for (int k = 0; k < 4; ++k) atomicMax(&info[4 * (size_t)tile + k], v[k]);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < kSlots) {
        const uint32_t slot = threadIdx.x;
        const uint32_t tile = slot == 0 ? tile0 : tile1 + slot - 1u;
        if (tile < T && (slot == 0 || tile != tile0)) {
            if (s_acc[slot]) atomicAdd(&sums[tile], s_acc[slot]);
            if (s_rej[slot]) atomicAdd(&sums[Tp + tile], s_rej[slot]);
            // (plain stores: the blocks of a dense top cell do not wait for each other)
            for (uint32_t w = 0; w < 2u; ++w)
                if (s_open[slot][w]) info[(4 + w) * (size_t)T + tile] = 1u;
            if (s_info[slot][0])
                for (int k = 0; k < 4; ++k) atomicMax(&info[4 * (size_t)tile + k], s_info[slot][k]);
        }
    }
}

// the grand totals (accepted ta, rejected tr) and the header's leaf-pair counts
SG_D void leaf_totals(GridHeader* h, uint32_t status, const BuildArgs& a, uint32_t* __restrict__ sums, uint32_t T,
                      uint32_t ta, uint32_t tr) {
    const uint32_t Tp = leaf_sums_stride(T);
    const uint64_t total = (uint64_t)ta + tr;
    // top pairs that were cut off leave keys of no build: no tile gets a plan
    const bool cut = (status & ST_CAP_P1) != 0u;
    sums[2 * (size_t)Tp] = cut ? 0xFFFFFFFFu : ta;
    sums[2 * (size_t)Tp + 1] = cut ? 0xFFFFFFFFu : tr;
    h->need_P2 = (uint32_t)min(total, (uint64_t)0xFFFFFFFFu);
    if (total > a.cap_P2) {
        atomicOr(&h->status, ST_CAP_P2);
        h->P2 = a.cap_P2;
        h->P2_valid = min(ta, a.cap_P2);
    } else {
        h->P2 = (uint32_t)total;
        h->P2_valid = ta;
    }
}

// First the wide boxes k_leaf_count listed are counted into their tiles'
// totals, a box to a block, and the last block that ends does the rest (one
// block for all took 3.2 us a box: 947 boxes in 200 dense cells 3.02 ms, with
// kScanBlocks of them 37 us; without wide boxes every block but the first
// leaves at once).  Then the exclusive scan, in place, of the accepted
// (sums[0..T)) and rejected (sums[Tp..Tp+T)) tile totals, both halves at once
// (waves 0-7 and 8-15); sums[2Tp], sums[2Tp+1] receive the grand totals and
// the header the leaf-pair counts (by one block of 1024 threads).
constexpr uint32_t kScanBlocks = 128;
__global__ __launch_bounds__(1024) void k_leaf_scan(TriSoA t, GridHeader* h, BuildArgs a,
                                                    const uint32_t* __restrict__ top_keys,
                                                    const uint32_t* __restrict__ top_vals,
                                                    const uint32_t* __restrict__ ranges,
                                                    const uint32_t* __restrict__ cells, uint32_t* sums,
                                                    uint32_t T) {
    constexpr int kPer = 16;
    __shared__ uint32_t s_w[16];
    __shared__ uint32_t s_tot[2], s_tiles;
    __shared__ float s_tab[3][kAxisMax];
    __shared__ bool s_last;
    const uint32_t Tp = leaf_sums_stride(T);
    const uint32_t status = h->status, n_wide = min(sums[2 * (size_t)Tp + 2], kWideCap);
    if (n_wide) {
        const LeafParams L = read_leaf_params(h);
        for (uint32_t k = blockIdx.x; k < n_wide; k += gridDim.x) {
            const uint32_t i = sums[2 * (size_t)Tp + 4 + k], key = top_keys[i];
            LeafSetup st;
            const uint32_t c = leaf_pair(t, L, h, key, top_vals[i], cells, st);
            const uint32_t acc = wide_count<16>(L, st, s_tab, s_w);
            if (threadIdx.x == 0) {
                const uint32_t tile = reinterpret_cast<const uint2*>(ranges)[key].x / kLeafTile;
                if (tile < T) {
                    atomicAdd(&sums[tile], acc);
                    atomicAdd(&sums[Tp + tile], c - acc);
                }
            }
        }
        if (threadIdx.x == 0) {
            __threadfence();
            s_last = atomicAdd(&sums[2 * (size_t)Tp + 3], 1u) == gridDim.x - 1u;
        }
        __syncthreads();
        if (!s_last) return;
        __threadfence();   // the other blocks' totals
    } else if (blockIdx.x) {
        return;
    }
    const int w = wave_id(), half = w >> 3;
    const uint32_t tt = threadIdx.x & 511u;
    uint32_t* row = sums + (size_t)half * Tp;
    uint32_t run = 0, tiles = 0;   // tiles: those with pairs
    if (threadIdx.x == 0) s_tiles = 0;
    for (uint32_t c0 = 0; c0 < T; c0 += 512u * kPer) {
        const uint32_t i0 = c0 + tt * kPer;
        uint32_t v[kPer], sum = 0;
        if (i0 + kPer <= Tp) {
#pragma unroll
            for (int q = 0; q < kPer / 4; ++q) {
                const uint4 x = reinterpret_cast<const uint4*>(row + i0)[q];
                v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < kPer; ++k) v[k] = 0;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            if (i0 + k >= T) v[k] = 0;
            sum += v[k];
            tiles += v[k] ? 1u : 0u;
        }
        const uint32_t inc = wave_incl_scan(sum);
        if (lane_id() == 63) s_w[w] = inc;
        __syncthreads();
        uint32_t pre = 0, tot = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t x = s_w[8 * half + j];
            pre += (8 * half + j < w) ? x : 0u;
            tot += x;
        }
        __syncthreads();
        uint32_t p = run + pre + inc - sum;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t x = v[k];
            v[k] = p;
            p += x;
        }
        if (i0 + kPer <= Tp) {   // rows are padded to whole groups of kPer
#pragma unroll
            for (int q = 0; q < kPer / 4; ++q)
                reinterpret_cast<uint4*>(row + i0)[q] = make_uint4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        }
        run += tot;
    }
    if (tt == 0) s_tot[half] = run;
    tiles = wave_sum(tiles);
    if (half == 0 && lane_id() == 0) atomicAdd(&s_tiles, tiles);
    __syncthreads();
    if (threadIdx.x == 0) {
        leaf_totals(h, status, a, sums, T, s_tot[0], s_tot[1]);
        sums[2 * (size_t)Tp + 3] = s_tiles;
    }
}

// With per-pair totals (LeafLarge), in place of k_leaf_scan: the tile totals
// come from the scans of those, so that k_leaf_count's blocks need not add to
// the totals of one tile, a dense top cell's, in turn (507,000 pairs, with
// the scans side by side: rebuild 350 -> 329 us).  First the wide boxes k_leaf_count listed, a block each ...
__global__ __launch_bounds__(1024) void k_leaf_wide(TriSoA t, GridHeader* h, const uint32_t* __restrict__ top_keys,
                                                    const uint32_t* __restrict__ top_vals,
                                                    const uint32_t* __restrict__ cells,
                                                    const uint32_t* __restrict__ sums, uint32_t T,
                                                    uint32_t* __restrict__ pacc, uint32_t* __restrict__ prej) {
    __shared__ uint32_t s_w[16];
    __shared__ float s_tab[3][kAxisMax];
    const uint32_t* list = sums + 2 * (size_t)leaf_sums_stride(T) + 2;
    const uint32_t n_wide = min(list[0], kWideCap);
    if (blockIdx.x >= n_wide) return;
    const LeafParams L = read_leaf_params(h);
    for (uint32_t k = blockIdx.x; k < n_wide; k += gridDim.x) {
        const uint32_t i = list[2 + k];
        LeafSetup st;
        const uint32_t c = leaf_pair(t, L, h, top_keys[i], top_vals[i], cells, st);
        const uint32_t acc = wide_count<16>(L, st, s_tab, s_w);
        if (threadIdx.x == 0) {
            pacc[i] = acc;
            prej[i] = c - acc;
        }
    }
}

// ... then, from the exclusive scans of the per-pair totals, the totals before
// each tile: those before the first top cell that starts at or after pair
// kLeafTile * tile.
__global__ __launch_bounds__(kBlock) void k_leaf_tile_sums(GridHeader* h, BuildArgs a,
                                                           const uint32_t* __restrict__ top_keys,
                                                           const uint32_t* __restrict__ ranges,
                                                           const uint32_t* __restrict__ pacc,
                                                           const uint32_t* __restrict__ prej,
                                                           const uint32_t* __restrict__ sacc,
                                                           const uint32_t* __restrict__ srej,
                                                           uint32_t* __restrict__ sums, uint32_t T) {
    const uint32_t P1v = min(h->P1_valid, a.cap_P1), C1 = h->C1, tile = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t ta = P1v ? sacc[P1v - 1u] + pacc[P1v - 1u] : 0u, tr = P1v ? srej[P1v - 1u] + prej[P1v - 1u] : 0u;
    if (tile == 0) leaf_totals(h, h->status, a, sums, T, ta, tr);
    if (tile >= T) return;
    uint32_t i = tile * kLeafTile;
    if (i < P1v) {
        const uint32_t key = top_keys[i];
        if (key < C1) {
            const uint2 rg = reinterpret_cast<const uint2*>(ranges)[key];
            if (rg.x != i) i = rg.y;
        }
    }
    sums[tile] = i < P1v ? sacc[i] : ta;
    sums[leaf_sums_stride(T) + tile] = i < P1v ? srej[i] : tr;
}

// Where tile b's pairs go: prefixes from k_leaf_scan, tile bounds and leaf
// key range from k_leaf_count, and who emits it.
enum LeafMode : uint32_t { LEAF_NONE, LEAF_SMALL, LEAF_BIG, LEAF_OVERSIZE };
struct LeafTilePlan {
    uint32_t a0, a1, pre_acc, pre_rej, acc, rej, tot_acc, kbase, span;
    LeafMode mode;
    bool simple;   // LEAF_SMALL: one window, one chunk, no stored boxes
};

SG_D void leaf_tile_plan(const BuildArgs& a, bool large, const uint32_t* __restrict__ sums,
                         const uint32_t* __restrict__ info, uint32_t T, uint32_t b, LeafTilePlan& q) {
    const uint32_t Tp = leaf_sums_stride(T);
    const uint32_t tot_acc = sums[2 * (size_t)Tp], tot_rej = sums[2 * (size_t)Tp + 1];
    q.mode = LEAF_NONE;
    if ((uint64_t)tot_acc + tot_rej > a.cap_P2) return;   // flagged by k_leaf_scan
    const uint4 inf = reinterpret_cast<const uint4*>(info)[b];
    if (inf.x == 0) return;   // no top cell starts in this tile
    q.a0 = ~inf.x;
    q.a1 = inf.y > q.a0 ? inf.y : q.a0;
    if (q.a0 >= q.a1) return;
    q.tot_acc = tot_acc;
    q.pre_acc = sums[b];
    q.pre_rej = sums[Tp + b];
    q.acc = (b + 1 < T ? sums[b + 1] : tot_acc) - q.pre_acc;
    q.rej = (b + 1 < T ? sums[Tp + b + 1] : tot_rej) - q.pre_rej;
    q.kbase = ~inf.z;
    q.span = inf.w >= q.kbase ? inf.w - q.kbase : 0xFFFFFFFFu;
    const uint32_t tops = q.a1 - q.a0;
    const bool stored = info[4 * (size_t)T + b] != 0u, wide = info[5 * (size_t)T + b] != 0u;
    const bool one = q.span <= LeafSmall::window && q.acc <= LeafSmall::chunk;
    q.simple = !stored && !wide && one;
    // a heavy tile among light ones is better cut in slices than left to a block
    // (sphere 160 against 141 us, ruins 275 against 236); where most are heavy, as
    // many blocks as tiles use the chip already (518,162-triangle height field, top
    // cells of 345 triangles: 208 against 287)
    auto heavy = [&]() {
        return q.acc > LeafSmall::chunk && 2ull * q.acc * sums[2 * (size_t)Tp + 3] > 3ull * tot_acc;
    };
    const bool small = (one || (!large && q.acc <= LeafSmall::pairs && q.span <= LeafSmall::span)) &&
                       tops <= LeafSmall::tops && !wide,
               big = !large && q.acc <= LeafBig::pairs && q.span <= LeafBig::span && tops <= LeafBig::tops;
    if (small && !(big && heavy())) q.mode = LEAF_SMALL;
    else if (big) q.mode = LEAF_BIG;
    else q.mode = LEAF_OVERSIZE;
}

// 16-bit counters in LDS, two to a word: add one, return the old value
SG_D uint32_t count_add(uint16_t* s_cnt, uint32_t k) {
    const uint32_t sh = (k & 1u) * 16u;
    return (atomicAdd(reinterpret_cast<uint32_t*>(s_cnt) + (k >> 1), 1u << sh) >> sh) & 0xFFFFu;
}

// Exclusive scan of s_cnt[0..span) in place by a block of NW waves, its total,
// and the
// ranges of the tile's leaf cells, which no other tile holds: {first, last+1}
// of its references, {0, 0} without (the leaf cells of empty top cells between
// the tile's are zero as well); n_ranges of them lie below C2.  W words, 2 W
// cells, per thread and round: one where a tile rarely takes two rounds (the
// ranges' stores are then contiguous; four cost the height field 1 %), four for
// larger tiles, whose rounds of two barriers took a tenth of their time.
template <int NW, int W>
SG_D uint32_t leaf_scan_counts(uint16_t* s_cnt, uint32_t span, uint32_t first, uint32_t* s_scan,
                           uint2* __restrict__ ranges, uint32_t n_ranges) {
    uint32_t* words = reinterpret_cast<uint32_t*>(s_cnt);
    uint32_t run = 0;
    for (uint32_t k0 = 0; k0 < span; k0 += NW * 128 * W) {
        const uint32_t k = k0 + 2u * W * threadIdx.x;
        uint32_t w[W], sum = 0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            w[j] = k + 2u * j < span ? words[(k >> 1) + j] : 0u;
            sum += (w[j] & 0xFFFFu) + (w[j] >> 16);
        }
        uint32_t agg;
        uint32_t p = run + block_excl_scan<NW>(sum, &agg, s_scan);
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const uint32_t c = k + 2u * j, n0 = w[j] & 0xFFFFu, n1 = w[j] >> 16, f = first + p;
            if (c < span) words[(k >> 1) + j] = p | (p + n0) << 16;
            if (c < n_ranges && c < span) ranges[c] = n0 ? make_uint2(f, f + n0) : make_uint2(0u, 0u);
            if (c + 1u < n_ranges && c + 1u < span)
                ranges[c + 1u] = n1 ? make_uint2(f + n0, f + n0 + n1) : make_uint2(0u, 0u);
            p += n0 + n1;
        }
        run += agg;
    }
    __syncthreads();
    return run;
}

// The lists of the tile's leaf cells, s_ord[end of cell k-1 .. end of cell k)
// with the ends in s_end (s_ord begins with cell k0, at place `base`), were
// filled by LDS atomics, so their order is any;
// the canonical order is top pairs ascending.  Entry j of the lists holds x =
// (leaf cell << kTopBits | top pair); its place among the tile's accepted pairs
// is the start of its cell's list and the number of smaller entries in it:
// as many LDS reads as the list is long, U in flight, all lanes at once (a
// height field's lists hold 10 on average; sorting them in place, a lane or a
// wave to a list, left the other lanes waiting: 27 % of the kernel).  Lists
// beyond kLongList are sorted first, by leaf_sort_long.
constexpr uint32_t kLongList = 192;
template <uint32_t U>
SG_D uint32_t leaf_place(const uint32_t* s_ord, const uint16_t* s_end, uint32_t x, uint32_t j, uint32_t k0,
                         uint32_t base) {
    const uint32_t k = x >> kTopBits;
    const uint32_t st = k > k0 ? s_end[k - 1] - base : 0u, en = s_end[k] - base;
    if (en - st > kLongList) return j;
    uint32_t rank = 0;
    for (uint32_t i = st; i < en; i += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = s_ord[min(i + u, en - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) rank += i + u < en && v[u] < x ? 1u : 0u;
    }
    return st + rank;
}

// a wave sorts each long list of the leaf cells [k0, k1) with a bitmap over the tile's top pairs (bm, the
// wave's own `words` words)
template <int NW>
SG_D void leaf_sort_long(uint32_t* s_ord, const uint16_t* s_end, uint32_t k0, uint32_t k1, uint32_t base, uint32_t* bm,
                         uint32_t words) {
    const uint32_t l = (uint32_t)lane_id();
    for (uint32_t c0 = k0; c0 < k1; c0 += NW * 64) {
        const uint32_t k = c0 + threadIdx.x;
        const uint32_t st = k < k1 && k > k0 ? s_end[k - 1] - base : 0u, n = k < k1 ? s_end[k] - base - st : 0u;
        for (uint64_t big = __ballot(n > kLongList); big; big &= big - 1) {
            const int L = __ffsll((long long)big) - 1;
            const uint32_t lst = (uint32_t)__builtin_amdgcn_readlane((int)st, L),
                           ln = (uint32_t)__builtin_amdgcn_readlane((int)n, L),
                           hi = (uint32_t)__builtin_amdgcn_readlane((int)k, L) << kTopBits;
            for (uint32_t w = l; w < words; w += 64) bm[w] = 0;
            __threadfence_block();
            for (uint32_t i = l; i < ln; i += 64) {
                const uint32_t v = s_ord[lst + i] & ((1u << kTopBits) - 1u);
                if ((v >> 5) < words) atomicOr(&bm[v >> 5], 1u << (v & 31u));
            }
            __threadfence_block();
            uint32_t run = lst;
            for (uint32_t w0 = 0; w0 < words; w0 += 64) {
                const uint32_t w = w0 + l;
                uint32_t m = w < words ? bm[w] : 0u;
                const uint32_t c = (uint32_t)__popc(m), inc = wave_incl_scan(c);
                uint32_t p = run + inc - c;
                for (; m; m &= m - 1u) s_ord[p++] = hi | (32u * w + (uint32_t)__ffs((int)m) - 1u);
                run += (uint32_t)__shfl((int)inc, 63, 64);
            }
            __threadfence_block();
        }
    }
    __syncthreads();
}

// the rejected pairs of one top pair, from slot r of the tail
SG_D void leaf_reject(uint32_t r, uint32_t n, uint32_t tri, uint32_t cap, uint32_t C2, uint32_t* __restrict__ keys,
                      uint32_t* __restrict__ vals, int write_keys) {
    for (; n && r < cap; --n, ++r) {
        if (write_keys) keys[r] = C2;
        vals[r] = tri;
    }
}

// Tiles that fit LeafSmall.  Each pair's box comes from k_leaf_count, so a
// tile is a counting sort of its accepted cells: LDS counts, one scan, LDS
// lists.  2,093,058-triangle height field, 6.6 M references: 140 us for 443 MB
// (3.2 TB/s; the reference records alone are 239 MB), VALU busy for half of
// it, the rest waiting for memory in the first loads (36 % of a block's time)
// and the write-out (40 %).  The form before it, a stable two-pass LDS radix
// sort of staged pairs with the boxes formed again from the gathered
// triangles, took 174 us.  Two pairs per lane in the write-out, so that their
// gathers overlap, changed nothing.
// A tile of more leaf cells than the LDS counts hold is sorted in windows of
// them, one of more pairs than the LDS lists hold in chunks of its counted
// cells (a cell's list is no longer than the tile's top pairs, so every chunk
// holds a cell); most tiles are one chunk of one window, without stored boxes
// (SIMPLE), whose boxes stay in registers.  (Left to k_leaf_emit_big, which counts
// a tile once per slice and has one block to a CU: 200,000 triangles of 5.8 M
// references, 4,900 to a tile, rebuild 1,805 us, as chunks 366; the same number
// with 32 leaf cells to a triangle 287 and, as windows, 135; a window of 4096
// cells instead of 8192 was up to 20 % slower there and 1 % faster on the height
// field.)
template <bool SIMPLE>
SG_D void leaf_emit_small(const LeafTilePlan& q, const uint2* __restrict__ boxes, const uint32_t* __restrict__ pool,
                          const TriSoA& t, uint32_t n_tris, uint32_t C1, uint32_t C2, uint32_t cap,
                          const uint32_t* __restrict__ top_keys, const uint32_t* __restrict__ top_vals,
                          const uint32_t* __restrict__ cells, uint32_t* __restrict__ keys,
                          uint32_t* __restrict__ vals, float* __restrict__ refs, uint32_t* __restrict__ leaves,
                          int write_keys, uint16_t* s_cnt, uint32_t* s_ord, uint32_t* s_tri, uint32_t* s_bm,
                          uint32_t* s_scan, uint32_t* s_k1) {
    constexpr int NW = kLeafBlock / 64;
    constexpr int R = LeafSmall::tops / kLeafBlock;   // rounds; a tile rarely needs more than two
    static_assert(LeafSmall::tops <= LeafSmall::chunk && LeafSmall::window <= 1u << (32 - kTopBits),
                  "a chunk holds a list, an entry a leaf cell of the window");
    const uint32_t tops = q.a1 - q.a0;
    uint32_t wn = min(q.span, LeafSmall::window);   // leaf cells of the window, from w0 on
    for (uint32_t k = threadIdx.x; 2u * k < wn; k += kLeafBlock) reinterpret_cast<uint32_t*>(s_cnt)[k] = 0;
    uint2 box[R];
    uint32_t at[R];   // the top cell's first leaf cell in the tile (16 bits), its resolution along x and y
    auto load = [&](uint32_t i, uint2& bx, uint32_t& a) {
        bx = make_uint2(kBoxEmpty, 0u);
        a = 0;
        if (i >= q.a1) return;
        const uint32_t key = top_keys[i];
        const uint2 y = boxes[i];
        if (key < C1) {
            const uint2 cl = reinterpret_cast<const uint2*>(cells)[key];
            bx = y;
            a = (cl.x - q.kbase) | cl.y << 16;
        }
    };
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const uint32_t i = q.a0 + (uint32_t)j * kLeafBlock + threadIdx.x;
        if (i < q.a1) s_tri[i - q.a0] = top_vals[i];
        if (SIMPLE) load(i, box[j], at[j]);
    }
    __syncthreads();
    // f(top pair, window's leaf cell) for the accepted cells of the window's
    // [k0, k1).  A simple tile's boxes stay in registers; the others' are read
    // again in each round, which needs no registers beyond the simple form's.
    auto over_tops = [&](uint32_t w0, uint32_t k0, uint32_t k1, auto&& f) {
        if (SIMPLE) {
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if ((uint32_t)j * kLeafBlock >= tops) break;
                box_visit(box[j], at[j] & 0xFFFFu, (at[j] >> 16) & 0xFFu, at[j] >> 24, [&](uint32_t k) {
                    if (k < k1) f((uint32_t)j * kLeafBlock + threadIdx.x, k);
                });
            }
            return;
        }
#pragma unroll 1
        for (uint32_t top = threadIdx.x; top < tops; top += kLeafBlock) {
            uint2 bx;
            uint32_t a, lo, hi;
            load(q.a0 + top, bx, a);
            if (bx.x == kBoxEmpty) continue;
            const uint32_t first = a & 0xFFFFu, crx = (a >> 16) & 0xFFu, cry = a >> 24;
            box_bounds(box_extent(bx, pool), first, crx, cry, lo, hi);
            if (hi < w0 + k0 || lo >= w0 + k1) continue;   // a box beside the cells has nothing there
            auto cell = [&](uint32_t k) {
                k -= w0;
                if (k - k0 < k1 - k0) f(top, k);
            };
            if (bx.x < kBoxOpen) box_visit(bx, first, crx, cry, cell);
            else stored_visit(bx, pool, first, crx, cry, cell);
        }
    };
    uint32_t done = q.pre_acc;   // the slot of the window's first pair
    for (uint32_t w0 = 0;;) {
        over_tops(w0, 0u, wn, [&](uint32_t, uint32_t k) { count_add(s_cnt, k); });
        if (w0 == 0u && q.rej) {
            uint32_t run = q.tot_acc + q.pre_rej;
            auto round = [&](uint32_t top, uint32_t n) {
                uint32_t agg;
                const uint32_t r = run + block_excl_scan<NW>(n, &agg, s_scan);
                if (n) leaf_reject(r, n, s_tri[top], cap, C2, keys, vals, write_keys);
                run += agg;
            };
            if (SIMPLE) {
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    if ((uint32_t)j * kLeafBlock >= tops) break;
                    round((uint32_t)j * kLeafBlock + threadIdx.x,
                          box_cells(box[j].x) - (uint32_t)__popc(box[j].y));
                }
            } else {
#pragma unroll 1
                for (uint32_t top = threadIdx.x; top - threadIdx.x < tops; top += kLeafBlock) {
                    uint2 bx;
                    uint32_t a;
                    load(q.a0 + top, bx, a);
                    round(top, box_rejects(bx, pool));
                }
            }
        }
        __syncthreads();
        const uint32_t acc = leaf_scan_counts<NW, SIMPLE ? 1 : 4>(s_cnt, wn, done, s_scan,
                                                     reinterpret_cast<uint2*>(leaves) + q.kbase + w0,
                                                     leaves && C2 > q.kbase + w0 ? C2 - q.kbase - w0 : 0u);
        // chunk: the leaf cells [k0, k1), their pairs from `base` on
        for (uint32_t k0 = 0, base = 0; base < acc;) {
            uint32_t k1 = wn, end = acc;
            if (!SIMPLE && acc - base > LeafSmall::chunk) {   // up to the first list that ends beyond the chunk
                for (uint32_t k = k0 + threadIdx.x; k < wn; k += kLeafBlock) {
                    const uint32_t en = k + 1u < wn ? s_cnt[k + 1u] : acc;
                    if (s_cnt[k] - base <= LeafSmall::chunk && en - base > LeafSmall::chunk) *s_k1 = k;
                }
                __syncthreads();
                k1 = *s_k1;
                end = s_cnt[k1];
                __syncthreads();
            }
            over_tops(w0, k0, k1, [&](uint32_t top, uint32_t k) {
                const uint32_t p = count_add(s_cnt, k) - base;
                if (p < LeafSmall::chunk) s_ord[p] = k << kTopBits | top;
            });
            __syncthreads();
            leaf_sort_long<NW>(s_ord, s_cnt, k0, k1, base, s_bm + LeafSmall::tops / 32 * wave_id(),
                               LeafSmall::tops / 32);
            // [0, end - base) of s_ord is filled: every accepted cell was counted and listed
            for (uint32_t j = threadIdx.x; j < end - base; j += kLeafBlock) {
                const uint32_t x = s_ord[j];
                if ((x >> kTopBits) >= wn) continue;
                const uint32_t idx = done + base + leaf_place<4>(s_ord, s_cnt, x, j, k0, base);
                const uint32_t tri = s_tri[min(x & ((1u << kTopBits) - 1u), tops - 1u)];
                if (idx >= cap) continue;
                if (write_keys) keys[idx] = q.kbase + w0 + (x >> kTopBits);
                vals[idx] = tri;
                write_ref_record(refs, idx, t.rec, tri, n_tris);
            }
            if (SIMPLE) return;
            k0 = k1;
            base = end;
            if (base < acc) __syncthreads();   // s_ord is free again
        }
        if (SIMPLE) return;
        done += acc;
        w0 += LeafSmall::window;
        if (w0 >= q.span) break;
        __syncthreads();   // the lists are read
        wn = min(q.span - w0, LeafSmall::window);
        for (uint32_t k = threadIdx.x; 2u * k < wn; k += kLeafBlock) reinterpret_cast<uint32_t*>(s_cnt)[k] = 0;
        __syncthreads();
    }
}

// items receives the work of the larger kernel (tile | slice << kSliceShift),
// *todo its number
__global__ __launch_bounds__(kLeafBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_leaf_emit(
    TriSoA t, GridHeader* h, BuildArgs a, const uint32_t* __restrict__ top_keys, const uint32_t* __restrict__ top_vals,
    const uint32_t* __restrict__ cells, const uint2* __restrict__ boxes, const uint32_t* __restrict__ pool,
    uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, float* __restrict__ refs,
    const uint32_t* __restrict__ sums, const uint32_t* __restrict__ info, uint32_t T, uint32_t* __restrict__ leaves,
    int write_keys, int large, uint32_t* __restrict__ todo, uint32_t* __restrict__ items) {
    constexpr int NW = kLeafBlock / 64;
    __shared__ uint32_t s_scan[NW], s_ord[LeafSmall::chunk], s_tri[LeafSmall::tops], s_k1;
    __shared__ uint32_t s_bm[LeafSmall::tops / 32 * NW];
    __shared__ __align__(4) uint16_t s_cnt[LeafSmall::window];
    LeafTilePlan q;
    leaf_tile_plan(a, large != 0, sums, info, T, blockIdx.x, q);
    if (q.mode != LEAF_SMALL) {
        // too many leaf pairs: no tile has a plan, and the ranges would be
        // those of an earlier build
        if (q.mode == LEAF_NONE && leaves && (h->status & ST_CAP_P2)) clear_leaves(leaves, a.cap_C2);
        // oversize tiles of a grid with the parallel emission are its
        const uint32_t n = q.mode == LEAF_BIG ? max(1u, (q.acc + kLeafSlice - 1u) / kLeafSlice)
                                              : (q.mode == LEAF_OVERSIZE && !large ? 1u : 0u);
        if (threadIdx.x == 0 && n) {
            const uint32_t at = atomicAdd(todo, n);
            for (uint32_t j = 0; j < n; ++j) items[at + j] = blockIdx.x | j << kSliceShift;
        }
        return;
    }
    if (q.simple)
        leaf_emit_small<true>(q, boxes, pool, t, h->n_tris, h->C1, h->C2, a.cap_P2, top_keys, top_vals, cells, keys,
                              vals, refs, leaves, write_keys, s_cnt, s_ord, s_tri, s_bm, s_scan, &s_k1);
    else
        leaf_emit_small<false>(q, boxes, pool, t, h->n_tris, h->C1, h->C2, a.cap_P2, top_keys, top_vals, cells, keys,
                               vals, refs, leaves, write_keys, s_cnt, s_ord, s_tri, s_bm, s_scan, &s_k1);
}

// One stable LSD pass by a block of kBigBlock threads over n (key, value)
// pairs in global memory: digit ((k - kbase) >> shift) & (2^db - 1), db <= 8,
// (k, v) -> (ko, vo).  Ranks as lds_sort_pass: a digit histogram, its scan,
// then rounds of kBigBlock pairs ranked by wave ballots and ordered across
// waves by per-wave digit counts.
SG_D void block_sort_pass_global(const uint32_t* k, const uint32_t* v, uint32_t* ko, uint32_t* vo, uint32_t n,
                                 uint32_t kbase, int shift, int db, uint32_t* s_base, uint32_t* s_wc,
                                 uint32_t* s_scan) {
    constexpr int NW = kBigBlock / 64;
    constexpr int RM = 256;
    const uint32_t R = 1u << db, mask = R - 1u;
    const int w = wave_id();
    const uint64_t lt = lanemask_lt();
    for (uint32_t j = threadIdx.x; j < RM * NW; j += kBigBlock) s_wc[j] = 0;
    if (threadIdx.x < RM) s_base[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kBigBlock) atomicAdd(&s_base[((k[i] - kbase) >> shift) & mask], 1u);
    __syncthreads();
    {
        const uint32_t c = threadIdx.x < R ? s_base[threadIdx.x] : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan<NW>(c, &tot, s_scan);
        if (threadIdx.x < R) s_base[threadIdx.x] = ex;
        __syncthreads();
    }
    for (uint32_t r0 = 0; r0 < n; r0 += kBigBlock) {
        const uint32_t i = r0 + threadIdx.x;
        const bool ok = i < n;
        const uint32_t x = ok ? k[i] : 0u, y = ok ? v[i] : 0u;
        const uint32_t d = ((x - kbase) >> shift) & mask;
        const uint64_t peers = digit_peers(ok, d, db);
        const uint32_t rk = (uint32_t)__popcll(peers & lt);
        if (ok && rk == 0) s_wc[w * RM + d] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (ok) {
            uint32_t pos = s_base[d] + rk;
            for (int u = 0; u < w; ++u) pos += s_wc[u * RM + d];
            ko[pos] = x;
            vo[pos] = y;
        }
        __syncthreads();
        if (threadIdx.x < R) {
            uint32_t c = 0;
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                c += s_wc[u * RM + threadIdx.x];
                s_wc[u * RM + threadIdx.x] = 0;
            }
            s_base[threadIdx.x] += c;
        }
        __syncthreads();
    }
}

// LDS of k_leaf_emit_big: a tile's counts and lists, or the digit counts of a
// tile sorted in global memory
struct BigLds {
    union {
        struct {
            uint32_t ord[kLeafSlice + LeafBig::tops];   // a list is no longer than the tile's top pairs
            uint16_t cnt[LeafBig::span];
        };
        struct {
            uint32_t base[256], wc[256 * (kBigBlock / 64)];
        };
    };
    union {
        uint32_t bm[LeafBig::tops / 32 * (kBigBlock / 64)];   // leaf_sort_long, after the lists are filled
        struct {
            uint32_t wide[kBigBlock], wacc[kBigBlock], wrej[kBigBlock], wcnt[kBigBlock];
        };
    };
    float tab[3][kAxisMax];
    uint32_t scan[kBigBlock / 64];
    uint32_t n_wide, k0, k1;
};

// A slice of a tile that fits LeafBig: as leaf_emit_small, its top pairs in
// rounds, open boxes visited again, wide ones by the block.  Slice 0 also
// writes the rejected pairs and the leaf ranges.  200,000-triangle sphere (12
// such tiles, the largest of 20,456 accepted pairs): one block per tile 147
// us, in slices of 4096 pairs 84 us; with a count pass that does not wait for
// LDS and fewer scan rounds 81 us (38,665-triangle ruins: rebuild 292 -> 274
// us), in slices of 1024 pairs 60 us.  The global
// sort and range passes that such tiles needed before took 130 us.
SG_D void leaf_emit_big(const LeafTilePlan& q, uint32_t slice, const LeafParams& L, GridHeader* h,
                        const uint2* __restrict__ boxes, const uint32_t* __restrict__ pool, const TriSoA& t,
                        uint32_t cap, const uint32_t* __restrict__ top_keys,
                        const uint32_t* __restrict__ top_vals, const uint32_t* __restrict__ cells,
                        uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, float* __restrict__ refs,
                        uint32_t* __restrict__ leaves, int write_keys, BigLds& s) {
    constexpr int NW = kBigBlock / 64;
    for (uint32_t k = threadIdx.x; 2u * k < q.span; k += kBigBlock) reinterpret_cast<uint32_t*>(s.cnt)[k] = 0;
    uint32_t run = q.tot_acc + q.pre_rej, k0 = 0, k1 = q.span, base = 0;
    if (threadIdx.x == 0) s.k0 = s.k1 = q.span;
    // One pass over the top pairs counts and writes the rejected pairs, another
    // fills the lists; apart, so that the first adds without waiting for the
    // old counts.
    auto over_tops = [&](auto list) {
        constexpr bool LIST = decltype(list)::value;
        for (uint32_t c0 = q.a0; c0 < q.a1; c0 += kBigBlock) {
            __syncthreads();
            if (threadIdx.x == 0) s.n_wide = 0;
            __syncthreads();
            const uint32_t i = c0 + threadIdx.x;
            uint32_t rej = 0, tri = 0;
            // a leaf cell of the tile that pair p lies in
            auto add = [&](uint32_t k, uint32_t p) {
                if (!LIST) {
                    if (k < q.span) count_add(s.cnt, k);
                } else if (k >= k0 && k < k1) {
                    const uint32_t at = count_add(s.cnt, k) - base;
                    if (at < kLeafSlice + LeafBig::tops) s.ord[at] = k << kTopBits | (p - q.a0);
                }
            };
            if (i < q.a1) {
                const uint32_t key = top_keys[i];
                tri = top_vals[i];
                const uint2 box = key < L.C1 ? boxes[i] : make_uint2(kBoxEmpty, 0u);
                if (box.x == kBoxWide) {
                    LeafSetup st;
                    const uint32_t c = leaf_pair(t, L, h, key, tri, cells, st);
                    if (wide_box(L, st, c)) {
                        s.wide[atomicAdd(&s.n_wide, 1u)] = threadIdx.x;
                    } else if (c) {
                        leaf_visit(L, st, [&](uint32_t k, bool ok) {
                            if (ok) add(k - q.kbase, i);
                            else ++rej;
                        });
                    }
                } else if (box.x != kBoxEmpty) {
                    const uint2 cl = reinterpret_cast<const uint2*>(cells)[key];
                    // a box beside the slice has nothing to list
                    const uint32_t first = cl.x - q.kbase, crx = cl.y & 0xFFu, cry = (cl.y >> 8) & 0xFFu;
                    uint32_t lo, hi;
                    box_bounds(box_extent(box, pool), first, crx, cry, lo, hi);
                    if (!LIST || (hi >= k0 && lo < k1)) {
                        if (box.x < kBoxOpen) box_visit(box, first, crx, cry, [&](uint32_t k) { add(k, i); });
                        else stored_visit(box, pool, first, crx, cry, [&](uint32_t k) { add(k, i); });
                    }
                    if (!LIST) rej = box_rejects(box, pool);
                }
            }
            __syncthreads();
            const uint32_t n_wide = s.n_wide;
            for (uint32_t w = 0; w < n_wide; ++w) {
                const uint32_t p = c0 + s.wide[w];
                LeafSetup st;
                const uint32_t c = leaf_pair(t, L, h, top_keys[p], top_vals[p], cells, st);
                uint32_t acc = 0;
                wide_visit(L, st, s.tab, [&](uint32_t, uint32_t key0, int xa, int xb) {
                    for (int x = xa; x < xb; ++x) add(key0 + (uint32_t)x - q.kbase, p);
                    acc += (uint32_t)(xb - xa);
                });
                acc = block_sum<NW>(acc, s.scan);
                if (threadIdx.x == s.wide[w]) rej = c - acc;
            }
            if (LIST || slice || !q.rej) continue;
            uint32_t agg;
            const uint32_t r = run + block_excl_scan<NW>(rej, &agg, s.scan);
            run += agg;
            if (rej < kWideBox / 2) {
                leaf_reject(r, rej, tri, cap, L.C2, keys, vals, write_keys);
            } else {
                s.wacc[threadIdx.x] = r;
                s.wrej[threadIdx.x] = rej;
                s.wcnt[threadIdx.x] = tri;
            }
            // long runs of rejected pairs by the whole block
            __syncthreads();
            if (threadIdx.x == 0) s.n_wide = 0;
            __syncthreads();
            if (rej >= kWideBox / 2) s.wide[atomicAdd(&s.n_wide, 1u)] = threadIdx.x;
            __syncthreads();
            for (uint32_t w = 0; w < s.n_wide; ++w) {
                const uint32_t o = s.wide[w];
                for (uint32_t j = threadIdx.x; j < s.wrej[o]; j += kBigBlock)
                    leaf_reject(s.wacc[o] + j, 1u, s.wcnt[o], cap, L.C2, keys, vals, write_keys);
            }
        }
        __syncthreads();
    };
    over_tops(std::false_type{});
    leaf_scan_counts<NW, 4>(s.cnt, q.span, q.pre_acc, s.scan, reinterpret_cast<uint2*>(leaves) + q.kbase,
                         leaves && slice == 0 && L.C2 > q.kbase ? L.C2 - q.kbase : 0u);
    // the slice's leaf cells [k0, k1) and the place of its first pair
    for (uint32_t k = threadIdx.x; k < q.span; k += kBigBlock) {
        const uint32_t at = s.cnt[k], lo = slice * kLeafSlice, hi = lo + kLeafSlice;
        const bool start = k == 0u;
        const uint32_t before = start ? 0u : s.cnt[k - 1u];
        if (at >= lo && (start || before < lo)) s.k0 = k;
        if (at >= hi && (start || before < hi)) s.k1 = k;
    }
    __syncthreads();
    k0 = s.k0;
    k1 = s.k1;
    base = k0 < q.span ? s.cnt[k0] : q.acc;
    over_tops(std::true_type{});
    if (k0 >= k1) return;
    leaf_sort_long<NW>(s.ord, s.cnt, k0, k1, base, s.bm + LeafBig::tops / 32 * wave_id(), (q.a1 - q.a0 + 31u) / 32u);
    const uint32_t n = min((uint32_t)s.cnt[k1 - 1u] - base, kLeafSlice + LeafBig::tops);
    for (uint32_t j = threadIdx.x; j < n; j += kBigBlock) {
        const uint32_t x = s.ord[j];
        if ((x >> kTopBits) >= q.span) continue;
        const uint32_t idx = q.pre_acc + base + leaf_place<8>(s.ord, s.cnt, x, j, k0, base);
        const uint32_t tri = top_vals[min(q.a0 + (x & (LeafBig::tops - 1u)), q.a1 - 1u)];
        if (idx >= cap) continue;
        if (write_keys) keys[idx] = q.kbase + (x >> kTopBits);
        vals[idx] = tri;
        write_ref_record(refs, idx, t.rec, tri, L.n_tris);
    }
}

// An oversize tile of a grid without the parallel emission: the block emits
// the tile's pairs in emission order, sorts its accepted pairs (stable LSD
// passes over the tile-local key, ping-ponging with tk / tv) and writes their
// reference records and leaf ranges -- correct but slow, for a rebuild that
// meets an oversize tile the grid's build never met.
SG_D void leaf_emit_oversize(const LeafTilePlan& q, const LeafParams& L, GridHeader* h, const TriSoA& t, uint32_t cap,
                             const uint32_t* __restrict__ top_keys, const uint32_t* __restrict__ top_vals,
                             const uint32_t* __restrict__ cells, uint32_t* __restrict__ keys,
                             uint32_t* __restrict__ vals, uint32_t* __restrict__ tk, uint32_t* __restrict__ tv,
                             float* __restrict__ refs, uint32_t* __restrict__ leaves, BigLds& s_) {
    uint32_t *s_scan = s_.scan, *s_base = s_.base, *s_wc = s_.wc, *s_wide = s_.wide, *s_wacc = s_.wacc,
             *s_wrej = s_.wrej, *s_wcnt = s_.wcnt;
    uint32_t& s_nwide = s_.n_wide;
    float(*s_tab)[kAxisMax] = s_.tab;
    const uint32_t rej_base = q.tot_acc + q.pre_rej;
    if (threadIdx.x == 0) atomicAdd(&h->oversize, 1u);
    for (uint32_t k = threadIdx.x; k < q.span && q.span != 0xFFFFFFFFu; k += kBigBlock)
        if (q.kbase + k < L.C2) reinterpret_cast<uint2*>(leaves)[q.kbase + k] = make_uint2(0u, 0u);
    uint32_t run_acc = 0, run_rej = 0;
    for (uint32_t c0 = q.a0; c0 < q.a1; c0 += kBigBlock) {
        const uint32_t i = c0 + threadIdx.x;
        LeafSetup s;
        uint32_t tri = 0, c = 0, ca = 0;
        bool wide = false;
        if (threadIdx.x == 0) s_nwide = 0;
        __syncthreads();
        if (i < q.a1) {
            tri = top_vals[i];
            c = leaf_pair(t, L, h, top_keys[i], tri, cells, s);
            wide = wide_box(L, s, c);
            if (wide) s_wide[atomicAdd(&s_nwide, 1u)] = threadIdx.x;
            else if (c) leaf_visit(L, s, [&](uint32_t, bool ok) { ca += ok ? 1u : 0u; });
        }
        __syncthreads();
        const uint32_t nwide = s_nwide;
        for (uint32_t k = 0; k < nwide; ++k) {
            LeafSetup ws;
            const uint32_t pair = c0 + s_wide[k];
            leaf_pair(t, L, h, top_keys[pair], top_vals[pair], cells, ws);
            const uint32_t acc = wide_count<kBigBlock / 64>(L, ws, s_tab, s_scan);
            if (threadIdx.x == s_wide[k]) ca = acc;
        }
        uint32_t agg_a, agg_r;
        uint32_t pa = q.pre_acc + run_acc + block_excl_scan<kBigBlock / 64>(ca, &agg_a, s_scan);
        uint32_t pr = rej_base + run_rej + block_excl_scan<kBigBlock / 64>(c - ca, &agg_r, s_scan);
        if (wide) {
            s_wacc[threadIdx.x] = pa;
            s_wrej[threadIdx.x] = pr;
            s_wcnt[threadIdx.x] = ca;
        } else if (c) {
            leaf_visit(L, s, [&](uint32_t key, bool ok) {
                const uint32_t idx = ok ? pa++ : pr++;
                if (idx < cap) {
                    keys[idx] = ok ? key : L.C2;
                    vals[idx] = tri;
                }
            });
        }
        __syncthreads();
        for (uint32_t k = 0; k < nwide; ++k) {
            LeafSetup ws;
            const uint32_t w = s_wide[k], pair = c0 + w, wtri = top_vals[pair];
            const uint32_t wc = leaf_pair(t, L, h, top_keys[pair], wtri, cells, ws);
            wide_emit<kBigBlock / 64>(L, ws, s_tab, s_scan, wtri, s_wacc[w], s_wrej[w], wc - s_wcnt[w], cap, keys, vals);
        }
        __syncthreads();   // the lists are free for the next chunk
        run_acc += agg_a;
        run_rej += agg_r;
    }
    // the accepted pairs of this tile: [pre_acc, pre_acc + run_acc), keys in
    // [kbase, kbase + span) (leaf_tile_plan guarantees pre_acc + run_acc <= cap)
    __threadfence_block();
    __syncthreads();
    const uint32_t n = run_acc;
    uint32_t* k0 = keys + q.pre_acc;
    uint32_t* v0 = vals + q.pre_acc;
    uint32_t* k1 = tk + q.pre_acc;
    uint32_t* v1 = tv + q.pre_acc;
    const uint32_t span = q.span == 0xFFFFFFFFu ? 0xFFFFFFFFu : q.span;
    const int bits = 32 - __builtin_clz(span | 1u);
    const int passes = (bits + 7) / 8;
    const int db = (bits + passes - 1) / passes;
    for (int p = 0, lo = 0; p < passes; ++p, lo += db) {
        if (p & 1) block_sort_pass_global(k1, v1, k0, v0, n, q.kbase, lo, min(db, bits - lo), s_base, s_wc, s_scan);
        else block_sort_pass_global(k0, v0, k1, v1, n, q.kbase, lo, min(db, bits - lo), s_base, s_wc, s_scan);
        __threadfence_block();
        __syncthreads();
    }
    if (passes & 1) {
        for (uint32_t i = threadIdx.x; i < n; i += kBigBlock) {
            k0[i] = k1[i];
            v0[i] = v1[i];
        }
    }
    for (uint32_t i = threadIdx.x; i < n; i += kBigBlock)
        write_ref_record(refs, q.pre_acc + i, t.rec, (passes & 1) ? v1[i] : v0[i], L.n_tris);
    // the ranges of the tile's leaf cells from its sorted keys (as k_leaf_emit)
    __threadfence_block();
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kBigBlock) {
        const uint32_t key = k0[i];
        if (i == 0 || k0[i - 1] != key) leaves[2 * (size_t)key] = q.pre_acc + i;
        if (i + 1 == n || k0[i + 1] != key) leaves[2 * (size_t)key + 1] = q.pre_acc + i + 1u;
    }
}

// the work k_leaf_emit left, an item per block; most builds have none
constexpr uint32_t kBigBlocks = 256;
__global__ __launch_bounds__(kBigBlock) void k_leaf_emit_big(
    TriSoA t, GridHeader* h, BuildArgs a, const uint32_t* __restrict__ top_keys, const uint32_t* __restrict__ top_vals,
    const uint32_t* __restrict__ cells, const uint2* __restrict__ boxes, const uint32_t* __restrict__ pool,
    uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, float* __restrict__ refs,
    const uint32_t* __restrict__ sums, const uint32_t* __restrict__ info, uint32_t T, uint32_t* __restrict__ leaves,
    int write_keys, const uint32_t* __restrict__ todo, const uint32_t* __restrict__ items, uint32_t* __restrict__ tk,
    uint32_t* __restrict__ tv) {
    __shared__ BigLds s;
    const uint32_t n = min(*todo, kSlicesMax * T);
    if (blockIdx.x >= n) return;
    const LeafParams L = read_leaf_params(h);
    for (uint32_t o = blockIdx.x; o < n; o += gridDim.x) {
        LeafTilePlan q;
        const uint32_t item = items[o];
        leaf_tile_plan(a, false, sums, info, T, item & ((1u << kSliceShift) - 1u), q);
        __syncthreads();   // s is free again
        if (q.mode == LEAF_BIG)
            leaf_emit_big(q, item >> kSliceShift, L, h, boxes, pool, t, a.cap_P2, top_keys, top_vals, cells, keys, vals,
                          refs, leaves, write_keys, s);
        else if (q.mode == LEAF_OVERSIZE)
            leaf_emit_oversize(q, L, h, t, a.cap_P2, top_keys, top_vals, cells, keys, vals, tk, tv, refs, leaves, s);
    }
}

// Oversize tiles with one thread per top pair: pair i of tile t writes its
// accepted pairs from pre_acc(t) + (sacc[i] - sacc[first pair of t]) and its
// rejected ones likewise (sacc / srej: exclusive scans of the per-pair totals
// of k_leaf_count), so the output is leaf_emit_oversize's, in parallel -- a
// top cell of 500k pairs (a dense cluster) no longer runs on one block.
__global__ __launch_bounds__(kBlock) void k_leaf_emit_par(TriSoA t, GridHeader* h, BuildArgs a,
                                                          const uint32_t* __restrict__ top_keys,
                                                          const uint32_t* __restrict__ top_vals,
                                                          const uint32_t* __restrict__ ranges,
                                                          const uint32_t* __restrict__ cells,
                                                          uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                          const uint32_t* __restrict__ sums,
                                                          const uint32_t* __restrict__ info, uint32_t T,
                                                          const uint32_t* __restrict__ prej,
                                                          const uint32_t* __restrict__ sacc,
                                                          const uint32_t* __restrict__ srej) {
    __shared__ uint32_t s_scan[kBlock / 64], s_wide[kBlock], s_nwide;
    __shared__ float s_tab[3][kAxisMax];
    const LeafParams L = read_leaf_params(h);
    const uint32_t P1v = min(h->P1_valid, a.cap_P1);
    const bool listed = sums[2 * (size_t)leaf_sums_stride(T) + 2] <= kWideCap;   // k_leaf_wide_emit has the wide boxes
    for (uint32_t base = blockIdx.x * kBlock; base < P1v; base += gridDim.x * kBlock) {
        if (threadIdx.x == 0) s_nwide = 0;
        __syncthreads();
        // the tile plan of pair i, when its tile is this kernel's
        LeafTilePlan q;
        auto mine = [&](uint32_t key) {
            if (key >= L.C1) return false;
            const uint32_t tile = reinterpret_cast<const uint2*>(ranges)[key].x / kLeafTile;
            if (tile >= T) return false;
            leaf_tile_plan(a, true, sums, info, T, tile, q);
            return q.mode == LEAF_OVERSIZE;
        };
        auto acc_slot = [&](uint32_t i) { return q.pre_acc + (sacc[i] - sacc[q.a0]); };
        auto rej_slot = [&](uint32_t i) { return q.tot_acc + q.pre_rej + (srej[i] - srej[q.a0]); };
        const uint32_t i = base + threadIdx.x;
        const uint32_t key = i < P1v ? top_keys[i] : L.C1;
        if (mine(key)) {
            if (i == q.a0) {
                h->leaf_sort = q.tot_acc;
                atomicAdd(&h->oversize, 1u);
            }
            const uint32_t tri = top_vals[i];
            LeafSetup s;
            const uint32_t c = leaf_pair(t, L, h, key, tri, cells, s);
            if (wide_box(L, s, c)) {
                if (!listed) s_wide[atomicAdd(&s_nwide, 1u)] = i;
            } else if (c) {
                uint32_t pa = acc_slot(i), pr = rej_slot(i);
                leaf_visit(L, s, [&](uint32_t k2, bool ok) {
                    const uint32_t idx = ok ? pa++ : pr++;
                    if (idx < a.cap_P2) {
                        keys[idx] = ok ? k2 : L.C2;
                        vals[idx] = tri;
                    }
                });
            }
        }
        __syncthreads();
        for (uint32_t k = 0; k < s_nwide; ++k) {
            const uint32_t w = s_wide[k], wkey = top_keys[w], wtri = top_vals[w];
            LeafSetup s;
            leaf_pair(t, L, h, wkey, wtri, cells, s);
            mine(wkey);
            wide_emit<kBlock / 64>(L, s, s_tab, s_scan, wtri, acc_slot(w), rej_slot(w), prej[w], a.cap_P2, keys, vals);
        }
        __syncthreads();   // the list is free for the next chunk
    }
}

// The wide boxes of oversize tiles, when k_leaf_count could list them all: one
// block of k_leaf_emit_par took 40 us for the 66,612 cells of one box, 63,000
// of them rejected.  While there are fewer of them than blocks, several blocks
// share a box: its rejected pairs, all alike, are split over them and the
// first emits the accepted ones.
constexpr uint32_t kWideBlocks = 64;
__global__ __launch_bounds__(1024) void k_leaf_wide_emit(TriSoA t, GridHeader* h, BuildArgs a,
                                                         const uint32_t* __restrict__ top_keys,
                                                         const uint32_t* __restrict__ top_vals,
                                                         const uint32_t* __restrict__ ranges,
                                                         const uint32_t* __restrict__ cells,
                                                         uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                         const uint32_t* __restrict__ sums,
                                                         const uint32_t* __restrict__ info, uint32_t T,
                                                         const uint32_t* __restrict__ prej,
                                                         const uint32_t* __restrict__ sacc,
                                                         const uint32_t* __restrict__ srej) {
    __shared__ uint32_t s_scan[16];
    __shared__ float s_tab[3][kAxisMax];
    const uint32_t* list = sums + 2 * (size_t)leaf_sums_stride(T) + 2;
    const uint32_t n = list[0];
    if (n == 0 || n > kWideCap) return;
    const uint32_t parts = max(1u, gridDim.x / n), part = blockIdx.x % parts;
    const LeafParams L = read_leaf_params(h);
    for (uint32_t k = blockIdx.x / parts; k < n; k += gridDim.x / parts) {
        const uint32_t i = list[2 + k], key = top_keys[i], tri = top_vals[i];
        const uint32_t tile = reinterpret_cast<const uint2*>(ranges)[key].x / kLeafTile;
        LeafTilePlan q;
        q.mode = LEAF_NONE;
        if (tile < T) leaf_tile_plan(a, true, sums, info, T, tile, q);
        if (q.mode != LEAF_OVERSIZE) continue;
        const uint32_t pr = q.tot_acc + q.pre_rej + (srej[i] - srej[q.a0]), rej = prej[i];
        for (uint32_t j = part * 1024u + threadIdx.x; j < rej; j += parts * 1024u)
            leaf_reject(pr + j, 1u, tri, a.cap_P2, L.C2, keys, vals, 1);
        if (part) continue;
        LeafSetup s;
        leaf_pair(t, L, h, key, tri, cells, s);
        wide_emit<16>(L, s, s_tab, s_scan, tri, q.pre_acc + (sacc[i] - sacc[q.a0]), 0u, 0u, a.cap_P2, keys, vals);
    }
}

// The global stable sort of the accepted leaf pairs works in two buffers;
// when its pass count is odd this copies its result back to the first one.
// n = GridHeader::leaf_sort, zero when every tile was sorted in LDS.
__global__ __launch_bounds__(kBlock) void k_copy_pairs(const uint32_t* __restrict__ ks,
                                                       const uint32_t* __restrict__ vs, uint32_t* __restrict__ kd,
                                                       uint32_t* __restrict__ vd, const uint32_t* d_n, uint32_t cap) {
    const uint32_t n = min(*d_n, cap);
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        kd[i] = ks[i];
        vd[i] = vs[i];
    }
}

// ---------------------------------------------------------------- launchers
static uint32_t init_blocks(const ZeroSegs& segs) {
    size_t total = 0;
    for (int i = 0; i < segs.count; ++i) total += segs.bytes[i] >> 4;
    uint32_t blocks = (uint32_t)((total + kBlock - 1) / kBlock);
    return blocks < 1 ? 1 : (blocks > 2048 ? 2048 : blocks);
}

static uint32_t ranges_blocks(uint32_t cap) {
    const uint32_t blocks = (cap + kBlock * 4 - 1) / (kBlock * 4);
    return blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks);
}

// one reference per thread (each record is a dependent gather)
static uint32_t refs_blocks(uint32_t cap) {
    const uint32_t blocks = (cap + kBlock - 1) / kBlock;
    return blocks < 1 ? 1 : (blocks > 32768 ? 32768 : blocks);
}

size_t bounds_blocks(uint32_t n) {
    const size_t b = ((size_t)n + kBlock * 4 - 1) / (kBlock * 4);   // 1024 triangles per block, four per lane
    return b < 1 ? 1 : (b > 4096 ? 4096 : b);
}

void launch_init_bounds(GridHeader* h, uint32_t n_tris, const ZeroSegs& segs, const TriSoA& t, uint32_t* part,
                        hipStream_t st) {
    const uint32_t nb = (uint32_t)bounds_blocks(n_tris);
    const uint32_t zb = init_blocks(segs);
    hipLaunchKernelGGL(k_init_bounds, dim3(nb > zb ? nb : zb), dim3(kBlock), 0, st, h, n_tris, segs, t, part, nb);
}

void launch_params(GridHeader* h, const BuildArgs& a, const uint32_t* part, uint32_t n, bool derive,
                   hipStream_t st) {
    hipLaunchKernelGGL(k_params, dim3(1), dim3(kBlock), 0, st, h, a, part, (uint32_t)bounds_blocks(n),
                       derive ? 1 : 0);
}

void launch_top_emit(const TriSoA& t, uint32_t n, GridHeader* h, const BuildArgs& a, const uint32_t* part,
                     uint32_t* keys, uint32_t* vals, uint32_t* dbg, uint32_t* sums, hipStream_t st) {
    const int items = top_items(n);
    const dim3 blocks((uint32_t)top_tiles(n, items)), tb(kBlock);
    if (n == 0) return;
    if (items == 1) {
        hipLaunchKernelGGL(k_top_count_params, blocks, tb, 0, st, t, n, h, a, part, (uint32_t)bounds_blocks(n), sums,
                           dbg);
        hipLaunchKernelGGL(k_top_emit<1>, blocks, tb, 0, st, t, n, h, a, keys, vals, sums);
    } else {
        launch_params(h, a, part, n, true, st);
        hipLaunchKernelGGL(k_top_count<kItems>, blocks, tb, 0, st, t, n, h, sums, dbg);
        hipLaunchKernelGGL(k_top_emit<kItems>, blocks, tb, 0, st, t, n, h, a, keys, vals, sums);
    }
}

void launch_ranges(const uint32_t* keys, const uint32_t* d_n, uint32_t cap, const uint32_t* d_C,
                   uint32_t* cells, uint32_t* d_pvalid, hipStream_t st) {
    hipLaunchKernelGGL(k_ranges, dim3(ranges_blocks(cap)), dim3(kBlock), 0, st, keys, d_n, cap, d_C, cells,
                       d_pvalid);
}

void launch_leaf_cells(GridHeader* h, const BuildArgs& a, const uint32_t* ranges, uint32_t* cells,
                       uint32_t* dbg, uint32_t* sums, uint32_t* leaves, hipStream_t st) {
    const uint32_t blocks = (a.cap_C1 + kBlock - 1) / kBlock;
    if (blocks == 0) return;
    hipLaunchKernelGGL(k_leaf_cells_count, dim3(blocks), dim3(kBlock), 0, st, h, a, ranges, sums, dbg);
    // blocks enough to clear the leaf ranges of a flagged grid of few top cells
    hipLaunchKernelGGL(k_leaf_cells_write, dim3(blocks < 256u ? 256u : blocks), dim3(kBlock), 0, st, h, a, ranges,
                       cells, sums, leaves);
}

void launch_leaf_emit(const TriSoA& t, GridHeader* h, const BuildArgs& a, const uint32_t* top_keys,
                      const uint32_t* top_vals, const uint32_t* ranges, const uint32_t* cells, uint32_t* keys,
                      uint32_t* vals, uint32_t* tmp_keys, uint32_t* tmp_vals, float* refs, uint32_t* dbg,
                      uint32_t* sums, uint32_t* info, uint2* boxes, uint32_t* box_pool, const LeafLarge* large,
                      uint32_t* leaves, hipStream_t st) {
    const uint32_t T = (uint32_t)leaf_tiles(a.cap_P1);
    const uint32_t blocks = (a.cap_P1 + kBlock - 1) / kBlock;
    const BoxPool pool{box_pool, (uint32_t)(leaf_pool_words(a.cap_P2) / kPools)};
    uint32_t* pool_n = sums + 2 * (size_t)leaf_sums_stride(T) + 4 + kWideCap;   // see leaf_sums_words
    uint32_t* todo = pool_n + kPools * kPoolStride;
    if (blocks)
        hipLaunchKernelGGL(k_leaf_count, dim3(blocks), dim3(kBlock), 0, st, t, h, top_keys, top_vals, ranges, cells,
                           sums, info, T, dbg, boxes, pool, pool_n, large ? large->pacc : nullptr,
                           large ? large->prej : nullptr);
    if (large) {
        const uint32_t* in[2] = {large->pacc, large->prej};
        uint32_t* out[2] = {large->sacc, large->srej};
        hipLaunchKernelGGL(k_leaf_wide, dim3(kWideBlocks), dim3(1024), 0, st, t, h, top_keys, top_vals, cells, sums, T,
                           large->pacc, large->prej);
        launch_scan_two(in, out, a.cap_P1, large->scan_scratch, st);
        hipLaunchKernelGGL(k_leaf_tile_sums, dim3((T + kBlock - 1) / kBlock), dim3(kBlock), 0, st, h, a, top_keys,
                           ranges, large->pacc, large->prej, large->sacc, large->srej, sums, T);
    } else {
        hipLaunchKernelGGL(k_leaf_scan, dim3(kScanBlocks), dim3(1024), 0, st, t, h, a, top_keys, top_vals, ranges,
                           cells, sums, T);
    }
    // with `large`, the global sort and k_ranges need every key; without it
    // the tiles write the leaf ranges and the keys are kept for keep_debug
    uint32_t* lv = large ? nullptr : leaves;
    const int write_keys = (large || a.keep_debug) ? 1 : 0;
    hipLaunchKernelGGL(k_leaf_emit, dim3(T), dim3(kLeafBlock), 0, st, t, h, a, top_keys, top_vals, cells, boxes,
                       box_pool, keys, vals, refs, sums, info, T, lv, write_keys, large ? 1 : 0, todo, todo + 1);
    // With `large` every tile beyond one chunk is oversize: its pairs are sorted by
    // the global sort that runs anyway.  (200,000-triangle sphere, 8 / 16 leaf cells
    // to a triangle: 303 / 371 us with them in the larger kernel, 243 / 269 so.)
    if (!large)
        hipLaunchKernelGGL(k_leaf_emit_big, dim3(kBigBlocks), dim3(kBigBlock), 0, st, t, h, a, top_keys, top_vals,
                           cells, boxes, box_pool, keys, vals, refs, sums, info, T, lv, write_keys, todo, todo + 1,
                           tmp_keys, tmp_vals);
    if (large) {
        uint32_t pb = (a.cap_P1 + kBlock - 1) / kBlock;
        pb = pb < 1 ? 1 : (pb > 4096 ? 4096 : pb);
        hipLaunchKernelGGL(k_leaf_emit_par, dim3(pb), dim3(kBlock), 0, st, t, h, a, top_keys, top_vals, ranges, cells,
                           keys, vals, sums, info, T, large->prej, large->sacc, large->srej);
        hipLaunchKernelGGL(k_leaf_wide_emit, dim3(kWideBlocks), dim3(1024), 0, st, t, h, a, top_keys, top_vals, ranges,
                           cells, keys, vals, sums, info, T, large->prej, large->sacc, large->srej);
    }
}

void launch_leaf_sort_fixup(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, GridHeader* h, uint32_t cap,
                            int key_bits, int radix_bits, uint32_t* scratch, hipStream_t st) {
    launch_sort_pairs(k0, v0, k1, v1, &h->leaf_sort, cap, key_bits, radix_bits, scratch, st);
    if (sort_passes(key_bits, radix_bits) & 1) {
        uint32_t blocks = (cap + kBlock * 4 - 1) / (kBlock * 4);
        blocks = blocks < 1 ? 1 : (blocks > 2048 ? 2048 : blocks);
        hipLaunchKernelGGL(k_copy_pairs, dim3(blocks), dim3(kBlock), 0, st, k1, v1, k0, v0, &h->leaf_sort, cap);
    }
}

// d_gate (optional): nothing to do while *d_gate == 0 (two-level grids: the
// LDS-sorted leaf tiles wrote their records in k_leaf_emit; only a global
// leaf sort, GridHeader::leaf_sort > 0, leaves them to this pass)
SG_D void ref_records_body(const uint32_t* __restrict__ indices, const uint32_t* d_valid, const uint32_t* d_gate,
                           uint32_t cap, const float* __restrict__ rec, uint32_t n_tris, float* __restrict__ refs,
                           uint32_t bid, uint32_t nb) {
    if (d_gate && *d_gate == 0) return;
    const uint32_t n = min(*d_valid, cap);
    for (uint32_t i = bid * kBlock + threadIdx.x; i < n; i += nb * kBlock)
        write_ref_record(refs, i, rec, indices[i], n_tris);
}

__global__ __launch_bounds__(kBlock) void k_ref_records(const uint32_t* __restrict__ indices, const uint32_t* d_valid,
                                                        const uint32_t* d_gate, uint32_t cap,
                                                        const float* __restrict__ rec, uint32_t n_tris,
                                                        float* __restrict__ refs) {
    ref_records_body(indices, d_valid, d_gate, cap, rec, n_tris, refs, blockIdx.x, gridDim.x);
}

void launch_ref_records(const uint32_t* indices, const uint32_t* d_valid, const uint32_t* d_gate, uint32_t cap,
                        const float* rec, uint32_t n_tris, float* refs, hipStream_t st) {
    hipLaunchKernelGGL(k_ref_records, dim3(refs_blocks(cap)), dim3(kBlock), 0, st, indices, d_valid, d_gate, cap,
                       rec, n_tris, refs);
}

// cell words from the cell ranges: a wave reads 64 neighbouring ranges and
// writes their two words
SG_D void cell_words_body(const uint32_t* __restrict__ ranges, uint32_t C, uint4* __restrict__ words, uint32_t bid,
                          uint32_t nb) {
    if (C < kWordCells) return;   // never read
    const uint32_t pairs = (C + 63u) / 64u;
    for (uint32_t w = bid * (kBlock / 64) + (uint32_t)wave_id(); w < pairs; w += nb * (kBlock / 64)) {
        const uint32_t k = 64u * w + (uint32_t)lane_id();
        const uint2 rg = k < C ? reinterpret_cast<const uint2*>(ranges)[k] : make_uint2(0u, 0u);
        const uint32_t n = rg.y - rg.x;
        const uint64_t m1 = __ballot(n >= 1u), m2 = __ballot(n >= 2u), m3 = __ballot(n >= 3u), m4 = __ballot(n >= 4u);
        const int sh = lane_id() & 32;
        const uint32_t h1 = (uint32_t)(m1 >> sh);
        const uint32_t first = (uint32_t)__shfl((int)rg.x, sh + (h1 ? __ffs((int)h1) - 1 : 0), 64);
        if ((lane_id() & 31) == 0)
            words[2u * w + (sh ? 1u : 0u)] = make_uint4(h1, (uint32_t)(m2 >> sh), (uint32_t)(m3 >> sh),
                                                        (uint32_t)(m4 >> sh) ? first | kWordFull : first);
    }
}

// the last launch of a uniform build: reference records and cell words
__global__ __launch_bounds__(kBlock) void k_uniform_records(const uint32_t* __restrict__ indices,
                                                            const GridHeader* h, uint32_t cap,
                                                            const float* __restrict__ rec, uint32_t n_tris,
                                                            float* __restrict__ refs,
                                                            const uint32_t* __restrict__ ranges, uint32_t cap_C,
                                                            uint4* __restrict__ words) {
    cell_words_body(ranges, min(h->C1, cap_C), words, blockIdx.x, gridDim.x);
    ref_records_body(indices, &h->P1_valid, nullptr, cap, rec, n_tris, refs, blockIdx.x, gridDim.x);
}

void launch_uniform_records(const uint32_t* indices, const GridHeader* h, uint32_t cap, const float* rec,
                            uint32_t n_tris, float* refs, const uint32_t* ranges, uint32_t cap_C, uint4* words,
                            hipStream_t st) {
    hipLaunchKernelGGL(k_uniform_records, dim3(refs_blocks(cap)), dim3(kBlock), 0, st, indices, h, cap, rec, n_tris,
                       refs, ranges, cap_C, words);
}

// ------------------------------------------------ many uniform grids, one launch
// k_multi_*: one launch of a phase for every job of an entry table; each
// block runs the phase's body for its job (see UniJob)
// zeroing and bounds of every job in one launch, as k_init_bounds
__global__ __launch_bounds__(kBlock) void k_multi_init(const UniJob* __restrict__ jobs,
                                                       const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    init_body(j.h, j.n, j.z, bid, nb);
    if (bid < j.nb_bounds) {
        const TriSoA t = j.t;
        bounds_body(t, j.n, j.part, bid, j.nb_bounds);
    }
}

__global__ __launch_bounds__(kBlock) void k_multi_params(const UniJob* __restrict__ jobs,
                                                         const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const BuildArgs a = j.a;
    params_body(j.h, a, j.part, j.nb_bounds, 1);
}

__global__ __launch_bounds__(kBlock) void k_multi_top_count(const UniJob* __restrict__ jobs,
                                                            const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const TriSoA t = j.t;
    top_count_body<kItems>(t, j.n, j.h, j.sums, j.dbg, bid);
}

__global__ __launch_bounds__(kBlock) void k_multi_top_emit(const UniJob* __restrict__ jobs,
                                                           const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const TriSoA t = j.t;
    const BuildArgs a = j.a;
    top_emit_body<kItems>(t, j.n, j.h, a, j.k[0], j.v[0], j.sums, bid, nb);
}

__global__ __launch_bounds__(kBlock) void k_multi_ranges(const UniJob* __restrict__ jobs,
                                                         const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const int f = j.passes & 1;
    ranges_body(j.k[f], &j.h->P1, j.cap_P, &j.h->C1, j.ranges, &j.h->P1_valid, bid, nb);
}

__global__ __launch_bounds__(kBlock) void k_multi_refs(const UniJob* __restrict__ jobs,
                                                       const MultiEntry* __restrict__ e, uint32_t ne) {
    uint32_t bid, nb;
    const UniJob& j = jobs[multi_entry(e, ne, blockIdx.x, gridDim.x, bid, nb)];
    const int f = j.passes & 1;
    cell_words_body(j.ranges, min(j.h->C1, j.a.cap_C1), j.words, bid, nb);
    ref_records_body(j.v[f], &j.h->P1_valid, nullptr, j.cap_P, j.t.rec, j.n, j.refs, bid, nb);
}

uint32_t multi_blocks(const UniJob& j, MultiPhase ph) {
    switch (ph) {
        case MP_INIT: return init_blocks(j.z) > j.nb_bounds ? init_blocks(j.z) : j.nb_bounds;
        case MP_PARAMS: return 1;
        case MP_TOP_COUNT:
        case MP_TOP_EMIT: return (uint32_t)top_tiles(j.n, kItems);
        case MP_RANGES: return ranges_blocks(j.cap_P);
        case MP_REFS: return refs_blocks(j.cap_P);
        default: return 0;
    }
}

void launch_multi(MultiPhase ph, const UniJob* jobs, const MultiEntry* e, uint32_t ne, uint32_t blocks,
                  hipStream_t st) {
    if (ne == 0 || blocks == 0) return;
    const dim3 g(blocks), b(kBlock);
    switch (ph) {
        case MP_INIT: hipLaunchKernelGGL(k_multi_init, g, b, 0, st, jobs, e, ne); break;
        case MP_PARAMS: hipLaunchKernelGGL(k_multi_params, g, b, 0, st, jobs, e, ne); break;
        case MP_TOP_COUNT: hipLaunchKernelGGL(k_multi_top_count, g, b, 0, st, jobs, e, ne); break;
        case MP_TOP_EMIT: hipLaunchKernelGGL(k_multi_top_emit, g, b, 0, st, jobs, e, ne); break;
        case MP_RANGES: hipLaunchKernelGGL(k_multi_ranges, g, b, 0, st, jobs, e, ne); break;
        case MP_REFS: hipLaunchKernelGGL(k_multi_refs, g, b, 0, st, jobs, e, ne); break;
        default: break;
    }
}

// number of per-tile sums the emission kernels need for n items
size_t emit_tiles(uint32_t n) { return top_tiles(n, top_items(n)); }
size_t cell_tiles(uint32_t n) { return ((size_t)n + kBlock - 1) / kBlock; }
// leaf tiles over n sorted top pairs
size_t leaf_tiles(uint32_t n) {
    const size_t t = ((size_t)n + kLeafTile - 1) / kLeafTile;
    return t ? t : 1;
}
// accepted and rejected totals, their grand totals, the number of wide boxes and
// of k_leaf_scan's blocks that have ended (then of tiles with pairs), the list of wide boxes, the words used
// of the pool's parts, the number of work items of k_leaf_emit_big (all cleared
// before each build), then the items
size_t leaf_sums_words(uint32_t n) {
    return 2 * (size_t)leaf_sums_stride((uint32_t)leaf_tiles(n)) + 4 + kWideCap + kPools * kPoolStride + 1;
}
size_t leaf_item_words(uint32_t n) { return kSlicesMax * leaf_tiles(n); }
size_t leaf_info_words(uint32_t n) { return 6 * leaf_tiles(n); }
// words of the pool for n leaf pairs: a stored box of c > 32 cells takes at most
// 2 + (c + 31) / 32 <= c / 8 of them
size_t leaf_pool_words(uint32_t n) { return (((size_t)n / 8 + 4096) / kPools) * kPools; }


}  // namespace sg
