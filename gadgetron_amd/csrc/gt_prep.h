// gt_prep.h -- preprocess of the hot paths without host round trips: tile keys,
// entry bounds and work items are formed on the device, in one stream, and the
// host reads back the few counts it launches with once, at the end.
//
// The host formed the work items before (counts down, items up, a
// synchronisation each, beside those for the range flag and the pair count): a
// new 2D frame (192^2, 34 spokes, 16 coils, gridding included) took 266-279 us,
// 143 of them on the device, and 113 with a library sort of the keys (38 us of
// the 100 on the device: seven launches of a merge sort for 52,000 key slots, its
// radix passes 57 us).  Up to kSortSamples samples and kSortKeys tiles the keys
// are now put in order by counting, both binnings in the same launches: a chunk's
// tiles are counted where its keys are formed, the counts are summed over the
// chunks (count_prefix_kernel) and the tiles, and each chunk scatters its samples in order (scatter_kernel): 89 us, and
// 84 with items and tables in one launch (items_tables_kernel).  Preprocess alone,
// sorted by the library / by counting / in one launch with the tables, us: 13 k
// samples on 288^2 124 / 66 / 54, 66 k on 384^2 201 / 85 / 69, 262 k 378 / 165 / 130,
// 66 k on 768^2 216 / 175 / 116, 262 k 370 / 266 / 176.  Past the bounds the library's
// radix passes have enough work; there the entries are counted first, with a read-back
// more, so that the tables have their size and not that of the most tiles a window can
// touch (922 k samples on 512^2: 308 MB a plan against 516; 410 k on 768^2: 0.92 ms
// against 0.67).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gt_kernels_fast.h"

namespace gt {

// What the host needs to know of a binning, written to pinned host memory.
struct PrepCounts {
    int bad;         // trajectory out of range or not finite
    uint32_t n;      // entries
    int n_items, n_red, n_partials;
    int overflow;    // the item list did not fit its bound (a mistake in the bound)
};

// Tiles of 8 cells that a window touches along one dimension of a grid of at
// least 8 + KW cells: at most two, three where the last tile is short.
struct TileSpan {
    int t[3], n;
};
__device__ __forceinline__ TileSpan tile_span8(float p, const GridGeom& g, int d) {
    TileSpan s;
    const int lo = (int)ceilf(p - g.radius), hi = (int)floorf(p + g.radius);
    int cell = lo < 0 ? lo + g.nos[d] : (lo >= g.nos[d] ? lo - g.nos[d] : lo);
    int left = hi - lo + 1;
    s.n = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        s.t[i] = cell >> 3;
        if (left > 0) s.n = i + 1;
        const int len = min(8 - (cell & 7), g.nos[d] - cell);
        left -= len;
        cell += len;
        cell = cell >= g.nos[d] ? 0 : cell;
    }
    return s;
}

// Positions, range flag and keys of the 2D hot path, one thread a sample.
// raw: the caller's trajectory (null: pos holds the positions already).  wkeys: the
// sample's tiles in `slots` slots, unused ones with the key past the last (nkeys),
// which is no entry; hkeys / hvals: its home tile in the C2NC binning gh.  Null arrays
// are left out.
// Workgroup b takes samples [b chunk, (b + 1) chunk); wcnt / hcnt (or null) get its
// entries of every key at [b nkeys + key] and [b nhome + key], counted in LDS.
static __global__ __launch_bounds__(256) void prep2d_kernel(
    const float* __restrict__ raw, float* __restrict__ pos, long long nsamp, int chunk, long long M, GridGeom gw,
    GridGeom gh, uint32_t nkeys, uint32_t nhome, int slots, uint32_t* __restrict__ wkeys, uint32_t* __restrict__ hkeys, uint32_t* __restrict__ hvals, uint32_t* __restrict__ wcnt,
    uint32_t* __restrict__ hcnt, int* __restrict__ flag) {
    extern __shared__ uint32_t counts[];
    uint32_t* wc = counts;
    uint32_t* hc = counts + (wcnt ? nkeys : 0u);
    const uint32_t nc = (wcnt ? nkeys : 0u) + (hcnt ? nhome : 0u);
    if (nc) {
        for (uint32_t k = threadIdx.x; k < nc; k += 256) counts[k] = 0u;
        __syncthreads();
    }
    const long long j1 = min(nsamp, (long long)(blockIdx.x + 1) * chunk);
    for (long long j = (long long)blockIdx.x * chunk + threadIdx.x; j < j1; j += 256) {
        float p[2];
#pragma unroll
        for (int d = 0; d < 2; d++) {
            if (raw) {
                const float k = raw[2 * j + d];
                const bool ok = k >= -0.5f && k <= 0.5f;
                if (!ok) flag[0] = 1;
                // a position inside the grid either way: the call fails, after kernels that index by it
                p[d] = ok ? (k + 0.5f) * gw.nos_f[d] : 0.0f;
                pos[2 * j + d] = p[d];
            } else {
                p[d] = pos[2 * j + d];
            }
        }
        const uint32_t frame = (uint32_t)j / (uint32_t)M;
        if (wkeys) {
            const TileSpan sx = tile_span8(p[0], gw, 0), sy = tile_span8(p[1], gw, 1);
            const uint32_t base = frame * (uint32_t)gw.ntiles_total;
            int o = 0;
#pragma unroll
            for (int b = 0; b < 3; b++)
#pragma unroll
                for (int a = 0; a < 3; a++)
                    if (a < sx.n && b < sy.n && o < slots) {
                        const uint32_t key = base + (uint32_t)(sx.t[a] + gw.ntiles[0] * sy.t[b]);
                        wkeys[j * slots + o] = key;
                        if (wcnt) atomicAdd(&wc[key], 1u);
                        o++;
                    }
            for (; o < slots; o++) wkeys[j * slots + o] = nkeys;
        }
        if (hkeys) {
            float pw;
            const int tx = home_tile_1d(p[0], gh, 0, pw), ty = home_tile_1d(p[1], gh, 1, pw);
            const uint32_t key = frame * (uint32_t)gh.ntiles_total + (uint32_t)(tx + gh.ntiles[0] * ty);
            hkeys[j] = key;
            if (hvals) hvals[j] = (uint32_t)j;
            if (hcnt) atomicAdd(&hc[key], 1u);
        }
    }
    if (nc) {
        __syncthreads();
        if (wcnt)
            for (uint32_t k = threadIdx.x; k < nkeys; k += 256) wcnt[(size_t)blockIdx.x * nkeys + k] = wc[k];
        if (hcnt)
            for (uint32_t k = threadIdx.x; k < nhome; k += 256) hcnt[(size_t)blockIdx.x * nhome + k] = hc[k];
    }
}

// Bounds of the counting sort: tiles of both binnings together (a workgroup's
// counts, 4 bytes each, fill 64 KB of LDS at most) and samples (its chunks hold up
// to kSortChunk samples, kSortParts of them).
constexpr uint32_t kSortKeys = 16000;
constexpr int kSortParts = 256, kSortChunk = 1024;
constexpr long long kSortSamples = (long long)kSortParts * kSortChunk;

// One binning of the counting sort.  cnt: [part][key] entries, then their sums
// over the parts before.
struct CountSort {
    const uint32_t* keys;  // [sample][slot], at or past nkeys: no entry
    uint32_t* cnt;
    uint32_t* total;       // entries of each key
    uint32_t* start;       // first entry of each key, nkeys + 1
    uint32_t* list;        // sample of each entry
    uint32_t* sorted;      // key of each entry, or null
    uint32_t nkeys;
    int slots;
};

// Exclusive sums of cnt over the parts, for each key, and the totals: a workgroup
// takes 64 keys (the lanes), its 16 waves 1/16 of the parts each.  gridDim.y: the
// binnings.
static __global__ __launch_bounds__(1024) void count_prefix_kernel(CountSort a0, CountSort a1, int parts) {
    constexpr int kPer = kSortParts / 16;
    __shared__ uint32_t sums[16][64];
    const CountSort a = blockIdx.y ? a1 : a0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t k = blockIdx.x * 64 + lane;
    if (blockIdx.x * 64 >= a.nkeys) return;  // the whole workgroup
    uint32_t v[kPer], sum = 0;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int b = wave * kPer + i;
        v[i] = (k < a.nkeys && b < parts) ? a.cnt[(size_t)b * a.nkeys + k] : 0u;
        sum += v[i];
    }
    sums[wave][lane] = sum;
    __syncthreads();
    uint32_t run = 0, tot = 0;
    for (int w = 0; w < 16; w++) {
        const uint32_t x = sums[w][lane];
        if (w < wave) run += x;
        tot += x;
    }
    if (k >= a.nkeys) return;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int b = wave * kPer + i;
        if (b < parts) a.cnt[(size_t)b * a.nkeys + k] = run;
        run += v[i];
    }
    if (wave == 0) a.total[k] = tot;
}

// The entries of a part to their places: entry order within a key is that of the
// samples (a stable sort), so the binning does not depend on the launch.  Every
// workgroup sums the totals to the keys' first entries itself (the first one writes
// them out: one launch less than a scan of its own).  The first `waves` waves (as
// many as their counts fit 64 KB) take consecutive runs of the part, count their
// keys in LDS, and place 64 entries at a time, a lane after the lower lanes of the
// same key.  The latencies of the scan and of two passes over the part bound it.
// gridDim.y: the binnings.
static __global__ __launch_bounds__(256) void scatter_kernel(CountSort a0, CountSort a1, long long nsamp, int chunk,
                                                             int waves) {
    extern __shared__ uint32_t counts[];  // [wave][key]
    __shared__ uint32_t sums[4];
    const CountSort a = blockIdx.y ? a1 : a0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t nk = a.nkeys;
    // the keys' first entries (of all parts) to the first wave's counts
    for (uint32_t k = threadIdx.x; k < nk; k += 256) counts[k] = a.total[k];
    for (uint32_t k = nk + threadIdx.x; k < nk * waves; k += 256) counts[k] = 0u;
    __syncthreads();
    const uint32_t kper = (nk + 255) / 256, k0 = min(nk, threadIdx.x * kper), k1 = min(nk, k0 + kper);
    uint32_t own = 0;
    for (uint32_t k = k0; k < k1; k++) own += counts[k];
    uint32_t x = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) sums[wave] = x;
    __syncthreads();
    uint32_t at = x - own;
    for (int w = 0; w < wave; w++) at += sums[w];
    for (uint32_t k = k0; k < k1; k++) {
        const uint32_t c = counts[k];
        counts[k] = at;
        at += c;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        for (uint32_t k = threadIdx.x; k < nk; k += 256) a.start[k] = counts[k];
        if (threadIdx.x == 255) a.start[nk] = at;
        __syncthreads();
    }
    // of this part and its waves: wave w's counts go to the wave after it
    for (uint32_t k = threadIdx.x; k < nk; k += 256) counts[k] += a.cnt[(size_t)blockIdx.x * nk + k];
    const uint32_t e0 = (uint32_t)((long long)blockIdx.x * chunk) * (uint32_t)a.slots;
    const uint32_t e1 = (uint32_t)min(nsamp, (long long)(blockIdx.x + 1) * chunk) * (uint32_t)a.slots;
    const uint32_t per = (e1 - e0 + 64 * waves - 1) / (64 * waves) * 64;
    const uint32_t b = min(e1, e0 + wave * per), e = wave < waves ? min(e1, b + per) : b;
    uint32_t* mine = counts + (size_t)wave * nk;
    if (wave + 1 < waves)
        for (uint32_t i = b + lane; i < e; i += 64) {
            const uint32_t k = a.keys[i];
            if (k < nk) atomicAdd(&mine[nk + k], 1u);
        }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nk; k += 256) {
        uint32_t run = counts[k];
        for (int w = 1; w < waves; w++) counts[w * nk + k] = run += counts[w * nk + k];
    }
    __syncthreads();
    for (uint32_t i0 = b; i0 < e; i0 += 64) {  // uniform over the wave
        const uint32_t i = i0 + lane, k = i < e ? a.keys[i] : nk;
        const bool on = k < nk;
        unsigned long long same = __builtin_amdgcn_ballot_w64(on);
        for (uint32_t m = 1; m < nk; m <<= 1) {
            const unsigned long long set = __builtin_amdgcn_ballot_w64((k & m) != 0u);
            same &= (k & m) ? set : ~set;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1ull));
        uint32_t first = 0;
        if (on && rank == 0) first = atomicAdd(&mine[k], (uint32_t)__popcll(same));
        first = __shfl(first, on ? __ffsll((long long)same) - 1 : 0);
        if (on) {
            a.list[first + rank] = i / (uint32_t)a.slots;
            if (a.sorted) a.sorted[first + rank] = k;
        }
    }
}

// start[k] = first sorted entry of key k or above, k <= nkeys; sorted keys past
// nkeys - 1 (unused slots) count as nkeys.  Thread i fills the keys between its
// entry and the one before it.
static __global__ void key_starts_kernel(const uint32_t* __restrict__ keys, long long n, uint32_t nkeys,
                                         uint32_t* __restrict__ start) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    const uint32_t cur = i < n ? min(keys[i], nkeys) : nkeys;
    const long long prev = i > 0 ? (long long)min(keys[i - 1], nkeys) : -1;
    for (long long k = prev + 1; k <= (long long)cur; k++) start[k] = (uint32_t)i;
}

// Sums over the threads before this one of a workgroup of 1024, and over all.
struct ItemSums {
    unsigned long long work, parts;  // parts: split keys << 32 | their partials
    uint32_t items;
};
__device__ __forceinline__ ItemSums block_exclusive(ItemSums v, ItemSums* sh, ItemSums& tot) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    ItemSums x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long a = __shfl_up(x.work, o), b = __shfl_up(x.parts, o);
        const uint32_t c = __shfl_up(x.items, o);
        if (lane >= o) {
            x.work += a;
            x.parts += b;
            x.items += c;
        }
    }
    __syncthreads();
    if (lane == 63) sh[wave] = x;
    __syncthreads();
    ItemSums base{};
    tot = ItemSums{};
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const ItemSums y = sh[w];
        if (w < wave) {
            base.work += y.work;
            base.parts += y.parts;
            base.items += y.items;
        }
        tot.work += y.work;
        tot.parts += y.parts;
        tot.items += y.items;
    }
    return ItemSums{base.work + x.work - v.work, base.parts + x.parts - v.parts, base.items + x.items - v.items};
}

// One binning of items_tables_kernel's work items.
struct ItemArgs {
    const uint32_t* start;  // first entry of each key, nkeys + 1
    uint32_t nkeys;
    int len, lmin, lmax, partial;
    WorkItem* items;
    int cap;
    RedItem* red;
    PrepCounts* out;
};

// Work items of a binning from its entry bounds, by a workgroup of 1024 threads
// (the rules of make_items and xcd_order on the host): a key's entries are cut
// into segments of len (0: the largest power of two from lmin to lmax that
// leaves 2 items per CU), with partial tiles and their sums' list where partial
// is set (then empty tiles get an item too); the items go to `runs` runs of equal
// work in key order, each sorted longest first (in 64 length classes) and the
// runs interleaved.  The order of equal items within a class is left to atomics:
// it decides nothing but the launch order.
static __device__ __forceinline__ void make_items(const ItemArgs& a, int cus, int runs, const int* __restrict__ flag) {
    constexpr int kCls = 64, kRuns = 8, kNear = 8192;
    const uint32_t nkeys = a.nkeys;
    const bool partial = a.partial != 0;
    __shared__ int hist[kRuns * kCls];
    __shared__ ItemSums sh[16];
    __shared__ int rsize[kRuns];
    __shared__ unsigned long long bound[kRuns];  // work at which run g + 1 begins
    __shared__ uint32_t near_start[kNear + 1];
    const int t = threadIdx.x;
    const uint32_t per = (nkeys + 1023) / 1024;
    const uint32_t k0 = min(nkeys, (uint32_t)t * per), k1 = min(nkeys, k0 + per);
    const bool near = nkeys <= (uint32_t)kNear;  // the bounds are read from LDS
    const uint32_t n = a.start[nkeys];
    if (near) {
        for (uint32_t k = t; k <= nkeys; k += 1024) near_start[k] = a.start[k];
        __syncthreads();
    }
    auto start = [&](uint32_t k) -> uint32_t { return near ? near_start[k] : a.start[k]; };
    uint32_t L = (uint32_t)a.len;
    if (a.len == 0) {
        const uint32_t target = n / (uint32_t)(2 * max(cus, 1));
        L = (uint32_t)a.lmin;
        while (L * 2 <= min((uint32_t)a.lmax, target)) L *= 2;
    }
    auto segs = [&](uint32_t c) -> uint32_t { return c <= L ? (c == 0 && !partial ? 0u : 1u) : (c + L - 1) / L; };
    ItemSums own{};
    for (uint32_t k = k0; k < k1; k++) {
        const uint32_t c = start(k + 1) - start(k), m = segs(c);
        own.items += m;
        own.work += m ? c + 32ull * m : 0ull;
        if (partial && c > L) own.parts += (1ull << 32) + m;
    }
    ItemSums all;
    const ItemSums before = block_exclusive(own, sh, all);
    const int G = all.items < 32 ? 1 : runs;
    for (int i = t; i < kRuns * kCls; i += 1024) hist[i] = 0;
    if (t < G) bound[t] = (all.work * (unsigned)(t + 1) + (unsigned)G - 1) / (unsigned)G;
    __syncthreads();
    const float scale = float(kCls - 1) / float(L);
    // lengths count in whole chunks of 32 entries, which is what an NC2C item takes time
    // by: items of one chunk then keep about the key order, and neighbouring tiles, which
    // share 128-byte lines of the grid, are written close together (24 frames of 21
    // spokes on 384^2, 8 coils: 117 -> 105 us).  C2NC shows no difference.
    const uint32_t step = partial ? 32u : 1u;
    // every item of the thread's keys: run and length class
    auto each = [&](auto&& f) {
        unsigned long long cum = before.work;
        uint32_t ri = (uint32_t)(before.parts >> 32), pi = (uint32_t)before.parts;
        int g = 0;
        for (uint32_t k = k0; k < k1; k++) {
            const uint32_t b = start(k), c = start(k + 1) - b, s = segs(c);
            const bool split = partial && c > L;
            if (split) f(-1, 0, k, ri++, pi, s);
            for (uint32_t q = 0; q < s; q++) {
                const uint32_t m = min(L, c - q * L);
                while (g < G - 1 && cum >= bound[g]) g++;
                const uint32_t mr = min(L, (m + step - 1) & ~(step - 1));
                const int cls = kCls - 1 - min(kCls - 1, (int)(float(mr) * scale));
                f(g, cls, k, b + q * L, m, split ? pi++ : 0xffffffffu);
                cum += m + 32;
            }
        }
    };
    each([&](int g, int cls, uint32_t, uint32_t, uint32_t, uint32_t) {
        if (g >= 0) atomicAdd(&hist[g * kCls + cls], 1);
    });
    __syncthreads();
    if (t < kRuns * kCls) {  // one wave a run: its classes' first positions
        const int c = hist[t];
        int x = c;
#pragma unroll
        for (int o = 1; o < kCls; o <<= 1) {
            const int y = __shfl_up(x, o);
            if ((t & 63) >= o) x += y;
        }
        hist[t] = x - c;
        if ((t & 63) == 63) rsize[t >> 6] = x;
    }
    __syncthreads();
    int longest = 1;  // keep one launchable item
    for (int g = 0; g < G; g++) longest = max(longest, rsize[g]);
    const bool fits = (long long)longest * G <= a.cap;
    if (fits) {
        each([&](int g, int cls, uint32_t k, uint32_t x, uint32_t y, uint32_t z) {
            if (g < 0) {
                a.red[x] = RedItem{k, (int32_t)y, (int32_t)z, 0};
                return;
            }
            const int pos = atomicAdd(&hist[g * kCls + cls], 1);
            a.items[pos * G + g] = WorkItem{k, x, x + y, (int32_t)z};  // z: partial slot or -1
        });
        for (int i = t; i < longest * G; i += 1024)
            if (i / G >= rsize[i % G]) a.items[i] = WorkItem{0u, 0u, 0u, kNoopItem};
    }
    if (t == 0) {
        a.out->bad = flag ? flag[0] : 0;
        a.out->n = n;
        a.out->n_items = longest * G;
        a.out->n_red = (int)(all.parts >> 32);
        a.out->n_partials = (int)(uint32_t)all.parts;
        a.out->overflow = fits ? 0 : 1;
    }
}

// Tables of the two binnings, as items_tables_kernel forms them.
struct TableArgs {
    const float* pos;
    const uint32_t *list, *keys, *n;  // NC2C: samples and keys of the entries, their number
    float* wt;
    uint32_t* hd;
    GridGeom gw;
    float csc;
    unsigned blocks;
    const uint32_t* hlist;  // C2NC on the matrix cores: samples of the entries, hn of them
    long long hn;
    float* wtab;
    GridGeom gh;
    float sx, sy;
};

// Work items and weight tables in one launch, which all need no more than the
// sorted entries: workgroups [0, nb) form a binning's items each (one workgroup
// and 16 to 20 us of latency, whatever the work), the next w.blocks the NC2C
// table, and the rest the C2NC table of the matrix cores, behind the items: 16 us for
// 13 k samples (items and the NC2C table apart 25), 21 for 66 k (all three apart 39).
template <int KW>
__global__ __launch_bounds__(1024) void items_tables_kernel(ItemArgs a0, ItemArgs a1, unsigned nb, TableArgs w, int cus,
                                                            int runs, const int* __restrict__ flag) {
    if (blockIdx.x < nb) {
        make_items(blockIdx.x ? a1 : a0, cus, runs, flag);
        return;
    }
    const unsigned b = blockIdx.x - nb;
    if (b < w.blocks) {
        const long long e = (long long)b * 1024 + threadIdx.x;
        if (e < (long long)*w.n) nc2c_table2d_entry(e, w.pos, w.list, w.keys, w.gw, w.wt, w.hd, w.csc);
    } else {
        const long long e = (long long)(b - w.blocks) * 1024 + threadIdx.x;
        if (e < w.hn) c2nc_wtable2d_entry<KW>(e, w.pos, w.hlist, w.gh, w.sx, w.sy, w.wtab);
    }
}

}  // namespace gt
