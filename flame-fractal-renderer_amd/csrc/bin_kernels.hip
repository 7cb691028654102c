// Binned accumulation of count-only buffers: the walker kernel writes one
// record per plotted sample (the cell index) instead of an atomic add; these
// kernels sort the records by tile with a counting sort and add each tile's
// counts from LDS into the buffer with plain loads and stores.
//
// The reference adds one to the cell per plotted sample with a relaxed
// atomic (src/renderers/buffer_renderer.hpp:211-215).  Counts are integers,
// so any order of adding them gives the same buffer.  On this device
// scattered global atomics are resolved at the memory side at ~23 G/s
// whatever their scope; a buffer far beyond the LDS whose samples spread
// over more cells than an LDS cache holds is bound by that rate.  Records
// move at HBM bandwidth instead:
//   walker   writes 4 B per sample (kEmptyKey where nothing is plotted)
//   hist     reads the records, one tile histogram per block of records
//   colscan  per tile, the running sum of the blocks' counts (the block's
//            first slot in the tile's region) and the tile's total
//   tilescan exclusive scan of the tile totals (the tiles' regions)
//   scatter  re-reads each block in chunks, sorts a chunk by tile in LDS and
//            writes each tile's run of it to the tile's region (consecutive
//            lanes, consecutive addresses)
//   accum    per tile, one workgroup per chunk of up to 2^17 of the
//            tile's records: counts in LDS, then one add per cell (an
//            atomic one where chunks share the tile)
// A tile is kBinTileCells consecutive cells (dimension 0 fastest), whose
// u32 counts fit the LDS of one workgroup.
#include "bin_common.hpp"
#include "util_kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace ffr {

namespace {

constexpr int kBinBlock = 256;                       // lanes per workgroup
constexpr unsigned kBinEmpty = kEmptyKey;

// records each lane loads before it uses them (independent loads in flight)
constexpr int kBinUnroll = 8;

// hist[b * ntiles + t] = records of block b in tile t
__global__ void __launch_bounds__(kBinBlock)
    bin_hist_kernel(const unsigned *rec, unsigned long long n, unsigned long long per_block,
                    int tile_bits, int ntiles, unsigned *hist)
{
    extern __shared__ unsigned h[];
    for (int t = threadIdx.x; t < ntiles; t += blockDim.x)
        h[t] = 0;
    __syncthreads();
    const unsigned long long b0 = (unsigned long long)blockIdx.x * per_block;
    const unsigned long long b1 = b0 + per_block < n ? b0 + per_block : n;
    constexpr unsigned long long step = (unsigned long long)kBinBlock * kBinUnroll;
    for (unsigned long long i0 = b0 + threadIdx.x; i0 < b1; i0 += step) {
        unsigned c[kBinUnroll];
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j) {
            const unsigned long long i = i0 + (unsigned long long)j * kBinBlock;
            c[j] = i < b1 ? rec[i] : kBinEmpty;
        }
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j)
            if (c[j] != kBinEmpty)
                atomicAdd(&h[c[j] >> tile_bits], 1u);
    }
    __syncthreads();
    unsigned *row = hist + (size_t)blockIdx.x * (size_t)ntiles;
    for (int t = threadIdx.x; t < ntiles; t += blockDim.x)
        row[t] = h[t];
}

// column scan: for tile t, hist[b][t] becomes the records of tiles t in
// blocks before b (exclusive), total[t] the tile's records.  A workgroup
// takes kScanTiles neighbouring tiles (whole lines of a row) and splits the
// blocks among kScanParts groups of lanes: their sums, then the running
// sums from each part's start.  (A lane per tile walked all blocks one
// after another: 90 us for 4096 tiles of 1024 blocks, now 10.)
constexpr int kScanTiles = 32, kScanParts = 32;

__global__ void __launch_bounds__(kScanTiles * kScanParts)
    bin_colscan_kernel(unsigned *hist, int nblocks, int ntiles, unsigned *total)
{
    __shared__ unsigned part[kScanParts][kScanTiles];
    const int tx = (int)threadIdx.x & (kScanTiles - 1), ty = (int)threadIdx.x / kScanTiles;
    const int t = (int)blockIdx.x * kScanTiles + tx;
    const int per = (nblocks + kScanParts - 1) / kScanParts;
    const int b0 = ty * per, b1 = min(nblocks, b0 + per);
    unsigned *col = hist + t; // (read and written for t < ntiles only)
    unsigned sum = 0;
    if (t < ntiles)
        for (int b = b0; b < b1; b += kBinUnroll) {
            unsigned v[kBinUnroll];
#pragma unroll
            for (int j = 0; j < kBinUnroll; ++j)
                v[j] = b + j < b1 ? col[(size_t)(b + j) * (size_t)ntiles] : 0u;
#pragma unroll
            for (int j = 0; j < kBinUnroll; ++j)
                sum += v[j];
        }
    part[ty][tx] = sum;
    __syncthreads();
    unsigned run = 0;
    for (int k = 0; k < kScanParts; ++k) {
        const unsigned v = part[k][tx];
        run += k < ty ? v : 0u;
    }
    if (t >= ntiles)
        return;
    if (ty == kScanParts - 1)
        total[t] = run + sum;
    for (int b = b0; b < b1; b += kBinUnroll) {
        unsigned v[kBinUnroll];
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j)
            v[j] = b + j < b1 ? col[(size_t)(b + j) * (size_t)ntiles] : 0u;
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j)
            if (b + j < b1) {
                col[(size_t)(b + j) * (size_t)ntiles] = run;
                run += v[j];
            }
    }
}

// exclusive scans over the tiles (one workgroup): of their records, into
// start[0..ntiles], and of their accumulation chunks of `chunk` records,
// into cstart[0..ntiles]
__global__ void __launch_bounds__(1024)
    bin_tilescan_kernel(const unsigned *total, int ntiles, unsigned chunk, unsigned *start,
                        unsigned *cstart)
{
    __shared__ unsigned part[1024], cpart[1024];
    const int tid = (int)threadIdx.x;
    const int per = (ntiles + (int)blockDim.x - 1) / (int)blockDim.x;
    const int t0 = tid * per;
    unsigned s = 0, c = 0;
    for (int k = 0; k < per; ++k)
        if (t0 + k < ntiles) {
            s += total[t0 + k];
            c += (total[t0 + k] + chunk - 1) / chunk;
        }
    part[tid] = s;
    cpart[tid] = c;
    __syncthreads();
    // Hillis-Steele inclusive scan of the per-thread sums
    for (int off = 1; off < (int)blockDim.x; off <<= 1) {
        const unsigned v = tid >= off ? part[tid - off] : 0u;
        const unsigned w = tid >= off ? cpart[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        cpart[tid] += w;
        __syncthreads();
    }
    unsigned run = tid ? part[tid - 1] : 0u, crun = tid ? cpart[tid - 1] : 0u;
    for (int k = 0; k < per; ++k)
        if (t0 + k < ntiles) {
            start[t0 + k] = run;
            cstart[t0 + k] = crun;
            run += total[t0 + k];
            crun += (total[t0 + k] + chunk - 1) / chunk;
        }
    if (tid == (int)blockDim.x - 1) {
        start[ntiles] = part[tid];
        cstart[ntiles] = cpart[tid];
    }
}

// Each block writes its records to their tiles' regions: the k-th record of
// tile t that block b writes goes to slot start[t] + hist[b][t] + k (the
// order inside a tile's region does not matter).  Written one by one from
// lanes holding records of many tiles, the 4-byte stores land on as many
// lines and reach HBM as partial writes (five times the record bytes were
// measured).  So the block takes its records in chunks of kScatterLanes x
// PER: a counting sort in LDS puts each chunk in tile order, and lane i then
// writes the chunk's i-th record, so that a tile's run of the chunk goes out
// from consecutive lanes to consecutive slots.
constexpr int kScatterLanes = 1024;

// LDS bytes of the scatter kernel for a tile count: the tiles' next slots,
// the chunk's counts per tile (offsets after the scan) and the chunk itself
// (whose first sixteen words hold the wave sums of the scan before it)
constexpr size_t scatter_lds(int ntiles, int per)
{
    return sizeof(unsigned) * (2 * (size_t)ntiles + (size_t)kScatterLanes * (size_t)per);
}

template <int PER>
__global__ void __launch_bounds__(kScatterLanes)
    bin_scatter_kernel(const unsigned *rec, unsigned long long n, unsigned long long per_block,
                       int tile_bits, int ntiles, const unsigned *hist, const unsigned *start,
                       unsigned *sorted)
{
    extern __shared__ unsigned lds[];
    unsigned *cur = lds;                   // [ntiles] next slot of each tile
    unsigned *off = cur + ntiles;          // [ntiles] chunk counts, then offsets
    unsigned *stage = off + ntiles;        // [kScatterLanes * PER] the chunk in tile order
    unsigned *wsum = stage;                // [16] wave sums of the scan (before the chunk)
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const unsigned *row = hist + (size_t)blockIdx.x * (size_t)ntiles;
    for (int t = tid; t < ntiles; t += kScatterLanes)
        cur[t] = start[t] + row[t];
    const unsigned long long b0 = (unsigned long long)blockIdx.x * per_block;
    const unsigned long long b1 = b0 + per_block < n ? b0 + per_block : n;
    constexpr unsigned long long chunk = (unsigned long long)kScatterLanes * PER;
    // tiles each lane scans (consecutive), at most 8 for 8192 tiles
    const int per_t = (ntiles + kScatterLanes - 1) / kScatterLanes;
    for (unsigned long long c0 = b0; c0 < b1; c0 += chunk) {
        for (int t = tid; t < ntiles; t += kScatterLanes)
            off[t] = 0;
        __syncthreads();
        // the chunk's records, counted per tile
        unsigned c[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const unsigned long long i = c0 + (unsigned long long)k * kScatterLanes + tid;
            c[k] = i < b1 ? rec[i] : kBinEmpty;
        }
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (c[k] != kBinEmpty)
                atomicAdd(&off[c[k] >> tile_bits], 1u);
        __syncthreads();
        // exclusive scan of the chunk's tile counts (per lane, then per
        // wave, then across the sixteen waves)
        const int t0 = tid * per_t;
        unsigned mine = 0;
        for (int j = 0; j < per_t; ++j)
            if (t0 + j < ntiles)
                mine += off[t0 + j];
        unsigned incl = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned y = __shfl_up(incl, d, 64);
            if (lane >= d)
                incl += y;
        }
        if (lane == 63)
            wsum[wave] = incl;
        __syncthreads();
        unsigned before = 0, total = 0;
        for (int w = 0; w < kScatterLanes / 64; ++w) {
            const unsigned ws = wsum[w];
            before += w < wave ? ws : 0u;
            total += ws; // the chunk's records
        }
        unsigned run = before + incl - mine;
        for (int j = 0; j < per_t; ++j)
            if (t0 + j < ntiles) {
                const unsigned v = off[t0 + j];
                off[t0 + j] = run;
                run += v;
            }
        __syncthreads(); // (the wave sums are read before the chunk overwrites them)
        // each record takes the next place of its tile's run; off[t] then
        // ends tile t's run, which begins where tile t - 1's ends
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (c[k] != kBinEmpty)
                stage[atomicAdd(&off[c[k] >> tile_bits], 1u)] = c[k];
        __syncthreads();
        for (unsigned i = (unsigned)tid; i < total; i += kScatterLanes) {
            const unsigned r = stage[i];
            const unsigned t = r >> tile_bits;
            sorted[cur[t] + (i - (t ? off[t - 1] : 0u))] = r;
        }
        __syncthreads();
        for (int t = tid; t < ntiles; t += kScatterLanes)
            cur[t] += off[t] - (t ? off[t - 1] : 0u);
        __syncthreads();
    }
}

// Tiles take very different shares of the records (the tetrahedron's
// lowest slices hold thousands of occupied cells, its highest a few), and
// one workgroup per tile left the device waiting on the largest.  So a tile
// is accumulated in chunks of at most `chunk` records (bin_accum_chunk), a
// workgroup each: the scan of their numbers gives tile t's work items
// cstart[t] .. cstart[t + 1].

// work item w: chunk w - cstart[t] of the tile t whose items hold w.  The
// chunk's counts go to LDS, then each cell's count into the buffer: a plain
// add when the tile has one chunk (no other workgroup touches it), an
// atomic one when several chunks share the tile.
template <typename CT>
__global__ void __launch_bounds__(1024)
    bin_accum_kernel(const unsigned *sorted, const unsigned *start, const unsigned *cstart,
                     int ntiles, int tile_bits, unsigned long long cells, unsigned chunk,
                     const unsigned *skip, CT *buf)
{
    extern __shared__ unsigned cnt[];
    const unsigned w = blockIdx.x;
    if (w >= cstart[ntiles] || (skip && *skip))
        return; // past the last work item (uniform across the workgroup)
    // the tile: the last t with cstart[t] <= w (tiles without records have
    // no items, so their cstart equals the next tile's)
    int lo = 0, hi = ntiles - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cstart[mid] <= w)
            lo = mid;
        else
            hi = mid - 1;
    }
    const int t = lo;
    const unsigned k = w - cstart[t];
    const bool shared = cstart[t + 1] - cstart[t] > 1;
    const unsigned s0 = start[t] + k * chunk;
    const unsigned s1 = min(start[t + 1], s0 + chunk);
    const unsigned tile = 1u << tile_bits;
    const unsigned long long c0 = (unsigned long long)t << tile_bits;
    const unsigned long long left = cells - c0;
    const unsigned ncell = left < tile ? (unsigned)left : tile;
    // (whole groups of 32: tile_word keeps a cell in its group)
    const unsigned nzero = (ncell + 31u) & ~31u;
    for (unsigned i = threadIdx.x; i < nzero; i += blockDim.x)
        cnt[i] = 0;
    __syncthreads();
    const unsigned mask = tile - 1u;
    const unsigned step = blockDim.x * (unsigned)kBinUnroll;
    for (unsigned i0 = s0 + threadIdx.x; i0 < s1; i0 += step) {
        unsigned c[kBinUnroll];
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j) {
            const unsigned i = i0 + (unsigned)j * blockDim.x;
            c[j] = i < s1 ? sorted[i] : kBinEmpty;
        }
#pragma unroll
        for (int j = 0; j < kBinUnroll; ++j)
            if (c[j] != kBinEmpty)
                atomicAdd(&cnt[tile_word(c[j] & mask)], 1u);
    }
    __syncthreads();
    for (unsigned i = threadIdx.x; i < ncell; i += blockDim.x) {
        const unsigned v = cnt[tile_word(i)];
        if (!v)
            continue;
        if (shared)
            atomicAdd(&buf[c0 + i], (CT)v);
        else
            buf[c0 + i] += (CT)v;
    }
}

// Colour flames: the scatter also moves each record's colour.  The walker
// leaves keys and colour components in arrays of their own; here a chunk's
// records are read once, put into tile order in LDS as whole records of NW
// words (key, colour, padding to 16 bytes) and written out as such, so that
// a tile's run of a chunk (8 records of 16 bytes for 1024 tiles) is one
// piece of memory.  The next chunk's records are read while this one is
// written.  (Moved one component at a time through LDS, with 4-byte runs
// and a barrier on every component's reads, a pass of 2^28 three-colour FP32
// records took 3.83 ms; now 2.67.)
constexpr size_t scatter_pay_lds(int ntiles, int per, int nw)
{
    return sizeof(unsigned) * ((size_t)nw * (size_t)kScatterLanes * (size_t)per +
                               2 * (size_t)ntiles + 16);
}

template <int PER, int NW, typename PR>
__global__ void __launch_bounds__(kScatterLanes)
    bin_scatter_pay_kernel(const unsigned *rec, const PR *pay, unsigned long long n,
                           unsigned long long per_block, int tile_bits, int ntiles,
                           const unsigned *hist, const unsigned *start, uint4 *sorted,
                           unsigned long long stride, int nr)
{
    constexpr int kReal = (int)sizeof(PR) / 4;
    constexpr int NR = (NW - 1) / kReal < 4 ? (NW - 1) / kReal : 4; // reals a record can hold
    constexpr int kChunk = kScatterLanes * PER;
    extern __shared__ uint4 stage[];                // [NW / 4][kChunk] records in tile order
    unsigned *cur = reinterpret_cast<unsigned *>(stage + NW / 4 * kChunk); // [ntiles] next slots
    unsigned *off = cur + ntiles;                   // [ntiles] chunk counts, then run starts
    unsigned *wsum = off + ntiles;                  // [16] wave sums of the scan
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const unsigned *row = hist + (size_t)blockIdx.x * (size_t)ntiles;
    for (int t = tid; t < ntiles; t += kScatterLanes) {
        cur[t] = start[t] + row[t];
        off[t] = 0;
    }
    const unsigned long long b0 = (unsigned long long)blockIdx.x * per_block;
    const unsigned long long b1 = b0 + per_block < n ? b0 + per_block : n;
    const int per_t = (ntiles + kScatterLanes - 1) / kScatterLanes;
    unsigned c[PER];
    PR v[PER][NR];
    auto load = [&](unsigned long long c0) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const unsigned long long i = c0 + (unsigned long long)k * kScatterLanes + tid;
            c[k] = i < b1 ? rec[i] : kBinEmpty;
#pragma unroll
            for (int j = 0; j < NR; ++j)
                if (j < nr)
                    v[k][j] = pay[(unsigned long long)j * stride + (i < b1 ? i : b0)];
        }
    };
    if (b0 < b1)
        load(b0);
    lds_barrier();
    for (unsigned long long c0 = b0; c0 < b1; c0 += kChunk) {
        // each record's rank in its tile's run of the chunk
        unsigned at[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k)
            at[k] = c[k] != kBinEmpty ? atomicAdd(&off[c[k] >> tile_bits], 1u) : 0u;
        lds_barrier();
        // exclusive scan of the chunk's tile counts (per lane, per wave,
        // across the sixteen waves)
        const int t0 = tid * per_t;
        unsigned mine = 0;
        for (int j = 0; j < per_t; ++j)
            if (t0 + j < ntiles)
                mine += off[t0 + j];
        unsigned incl = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned y = __shfl_up(incl, d, 64);
            if (lane >= d)
                incl += y;
        }
        if (lane == 63)
            wsum[wave] = incl;
        lds_barrier();
        unsigned before = 0, total = 0;
        for (int w = 0; w < kScatterLanes / 64; ++w) {
            const unsigned ws = wsum[w];
            before += w < wave ? ws : 0u;
            total += ws;
        }
        unsigned run = before + incl - mine;
        for (int j = 0; j < per_t; ++j)
            if (t0 + j < ntiles) {
                const unsigned m = off[t0 + j];
                off[t0 + j] = run;
                run += m;
            }
        lds_barrier();
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (c[k] != kBinEmpty) {
                unsigned w[NW];
#pragma unroll
                for (int j = 0; j < NW; ++j)
                    w[j] = 0;
                w[0] = c[k];
#pragma unroll
                for (int j = 0; j < NR; ++j)
                    if (j < nr)
                        put_real<PR>(w + 1 + j * kReal, v[k][j]);
                const unsigned pos = off[c[k] >> tile_bits] + at[k];
#pragma unroll
                for (int q = 0; q < NW / 4; ++q)
                    stage[q * kChunk + pos] =
                        make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
            }
        if (c0 + kChunk < b1)
            load(c0 + kChunk);
        lds_barrier();
        for (unsigned i = (unsigned)tid; i < total; i += kScatterLanes) {
            const uint4 first = stage[i];
            const unsigned t = first.x >> tile_bits;
            uint4 *dst = sorted + (size_t)(cur[t] + (i - off[t])) * (NW / 4);
            dst[0] = first;
#pragma unroll
            for (int q = 1; q < NW / 4; ++q)
                dst[q] = stage[q * kChunk + i];
        }
        lds_barrier();
        // (the run of tile t ends where the next one's starts)
        for (int j = 0; j < per_t; ++j)
            if (t0 + j < ntiles) {
                const unsigned end = t0 + j + 1 < ntiles ? off[t0 + j + 1] : total;
                cur[t0 + j] += end - off[t0 + j];
            }
        lds_barrier();
        for (int t = tid; t < ntiles; t += kScatterLanes)
            off[t] = 0;
        lds_barrier();
    }
}

// Colour flames: a chunk's counts and colour sums in LDS (u32 counts, f64
// sums of the records' colours), then one add per word of each occupied
// cell: plain where the tile has one chunk, atomic where chunks share it.
// Colour sums come out in another order than the atomic path's per-sample
// adds, equal to the rounding of that order.  Several records of a lane are
// in flight (one at a time, 2.36 ms per 2^28 three-colour FP32 records;
// now 1.44).
constexpr int kColourTile = 1 << kBinTileBitsColour;
constexpr int kColourUnroll = 4;

template <typename CT, typename CR, typename PR, int NW>
__global__ void __launch_bounds__(1024)
    bin_accum_colour_kernel(const uint4 *sorted, int nr, const unsigned *start,
                            const unsigned *cstart, int ntiles, unsigned long long cells,
                            unsigned chunk, const unsigned *skip, CT *buf)
{
    constexpr int kReal = (int)sizeof(PR) / 4;
    constexpr int NR = (NW - 1) / kReal < 4 ? (NW - 1) / kReal : 4;
    extern __shared__ unsigned long long lds64[];
    double *col = reinterpret_cast<double *>(lds64);                 // [nr][kColourTile]
    unsigned *cnt = reinterpret_cast<unsigned *>(col + 4 * kColourTile); // [kColourTile]
    const unsigned w = blockIdx.x;
    if (w >= cstart[ntiles] || (skip && *skip))
        return;
    int lo = 0, hi = ntiles - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cstart[mid] <= w)
            lo = mid;
        else
            hi = mid - 1;
    }
    const int t = lo;
    const unsigned k = w - cstart[t];
    const bool shared = cstart[t + 1] - cstart[t] > 1;
    const unsigned s0 = start[t] + k * chunk;
    const unsigned s1 = min(start[t + 1], s0 + chunk);
    const unsigned long long c0 = (unsigned long long)t * kColourTile;
    const unsigned long long left = cells - c0;
    const unsigned ncell = left < (unsigned long long)kColourTile ? (unsigned)left : kColourTile;
    const unsigned nzero = (ncell + 31u) & ~31u;
    for (unsigned i = threadIdx.x; i < nzero; i += blockDim.x) {
        cnt[i] = 0;
        for (int j = 0; j < nr; ++j)
            col[j * kColourTile + i] = 0.0;
    }
    __syncthreads();
    constexpr unsigned mask = kColourTile - 1;
    for (unsigned i0 = s0 + threadIdx.x; i0 < s1; i0 += blockDim.x * kColourUnroll) {
        unsigned v[kColourUnroll][NW];
#pragma unroll
        for (int u = 0; u < kColourUnroll; ++u) {
            const unsigned i = i0 + (unsigned)u * blockDim.x;
            const uint4 *src = sorted + (size_t)(i < s1 ? i : i0) * (NW / 4);
#pragma unroll
            for (int q = 0; q < NW / 4; ++q) {
                const uint4 x = src[q];
                v[u][4 * q] = x.x;
                v[u][4 * q + 1] = x.y;
                v[u][4 * q + 2] = x.z;
                v[u][4 * q + 3] = x.w;
            }
        }
#pragma unroll
        for (int u = 0; u < kColourUnroll; ++u) {
            if (i0 + (unsigned)u * blockDim.x >= s1)
                break;
            const unsigned cw = tile_word(v[u][0] & mask);
            atomicAdd(&cnt[cw], 1u);
#pragma unroll
            for (int j = 0; j < NR; ++j)
                if (j < nr)
                    atomicAdd(&col[j * kColourTile + cw], get_real<PR>(&v[u][1 + j * kReal]));
        }
    }
    __syncthreads();
    const int words = 1 + nr;
    for (unsigned i = threadIdx.x; i < ncell; i += blockDim.x) {
        const unsigned cw = tile_word(i);
        const unsigned n = cnt[cw];
        if (!n)
            continue;
        CT *cell = buf + (c0 + i) * (unsigned long long)words;
        CR *colour = reinterpret_cast<CR *>(cell + 1);
        if (shared) {
            atomicAdd(cell, (CT)n);
            for (int j = 0; j < nr; ++j)
                unsafeAtomicAdd(&colour[j], (CR)col[j * kColourTile + cw]);
        } else {
            *cell += (CT)n;
            for (int j = 0; j < nr; ++j)
                colour[j] += (CR)col[j * kColourTile + cw];
        }
    }
}

constexpr size_t accum_colour_lds()
{
    return sizeof(double) * 4 * kColourTile + sizeof(unsigned) * kColourTile;
}

// the scatter's records a lane per chunk, by record words and tiles: what
// the LDS holds
constexpr int kScatterTiles = 3072; // tiles beside the larger chunks
constexpr int scatter_per(int nw, bool many) { return nw == 4 ? (many ? 4 : 8) : nw == 8 ? (many ? 2 : 4) : (many ? 1 : 2); }

// the colour kernels of a record size: scatter, then (with the work items
// known) accumulation
template <typename PR, int NW>
void launch_scatter_pay(const BinScratch &b, unsigned long long n, unsigned long long per,
                        int nblocks, int tile_bits, int ntiles, int r, hipStream_t s)
{
    auto go = [&](auto kern, int per_lane) {
        hipLaunchKernelGGL(kern, dim3(nblocks), dim3(kScatterLanes),
                           scatter_pay_lds(ntiles, per_lane, NW), s, b.rec, (const PR *)b.pay, n,
                           per, tile_bits, ntiles, b.hist, b.start, (uint4 *)b.pay_sorted,
                           b.capacity, r);
    };
    if (ntiles <= kScatterTiles)
        go(bin_scatter_pay_kernel<scatter_per(NW, false), NW, PR>, scatter_per(NW, false));
    else
        go(bin_scatter_pay_kernel<scatter_per(NW, true), NW, PR>, scatter_per(NW, true));
}

template <typename PR, int NW>
void launch_accum_colour(const BinScratch &b, unsigned items, int r, const unsigned *cstart,
                         int ntiles, unsigned long long cells, unsigned chunk,
                         const unsigned *skip, void *buf, int word_bytes, hipStream_t s)
{
    // 8-byte words hold u64 counts and f64 sums, 4-byte words u32 and f32
    // (the float build); the records' colours are the walker's reals
    if (word_bytes == 8)
        hipLaunchKernelGGL((bin_accum_colour_kernel<unsigned long long, double, PR, NW>),
                           dim3(items), dim3(1024), accum_colour_lds(), s,
                           (const uint4 *)b.pay_sorted, r, b.start, cstart, ntiles, cells, chunk,
                           skip, (unsigned long long *)buf);
    else
        hipLaunchKernelGGL((bin_accum_colour_kernel<unsigned, float, PR, NW>), dim3(items),
                           dim3(1024), accum_colour_lds(), s, (const uint4 *)b.pay_sorted, r,
                           b.start, cstart, ntiles, cells, chunk, skip, (unsigned *)buf);
}

// f(a walker's real, the record's words) for a flame of r colours
template <typename F> void with_colour_record(int r, int real_bytes, F &&f)
{
    if (real_bytes == 8) {
        if (r <= 3)
            f(double(), std::integral_constant<int, record_words(3, 8)>());
        else
            f(double(), std::integral_constant<int, record_words(4, 8)>());
    } else {
        if (r <= 3)
            f(float(), std::integral_constant<int, record_words(3, 4)>());
        else
            f(float(), std::integral_constant<int, record_words(4, 4)>());
    }
}

template <typename PR, int NW> hipError_t prepare_colour()
{
    auto limit = [](const void *k, size_t bytes) {
        return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    };
    static_assert(scatter_pay_lds(kScatterTiles, scatter_per(NW, false), NW) <= 160 * 1024, "scatter chunk beyond the LDS");
    static_assert(scatter_pay_lds(kBinMaxTiles, scatter_per(NW, true), NW) <= 160 * 1024, "scatter chunk beyond the LDS");
    hipError_t e = limit((const void *)bin_scatter_pay_kernel<scatter_per(NW, false), NW, PR>,
                         scatter_pay_lds(kScatterTiles, scatter_per(NW, false), NW));
    if (e == hipSuccess)
        e = limit((const void *)bin_scatter_pay_kernel<scatter_per(NW, true), NW, PR>,
                  scatter_pay_lds(kBinMaxTiles, scatter_per(NW, true), NW));
    if (e == hipSuccess)
        e = limit((const void *)bin_accum_colour_kernel<unsigned long long, double, PR, NW>,
                  accum_colour_lds());
    if (e == hipSuccess)
        e = limit((const void *)bin_accum_colour_kernel<unsigned, float, PR, NW>,
                  accum_colour_lds());
    return e;
}

int grid_for(unsigned long long n, int block)
{
    unsigned long long g = (n + (unsigned long long)block - 1) / (unsigned long long)block;
    return (int)std::min<unsigned long long>(std::max<unsigned long long>(g, 1), 4096);
}

} // namespace

// records of a histogram and scatter block: 2^18, less for renders of few
// records, so that they spread over the device (about 512 blocks)
static unsigned long long bin_block_records(unsigned long long records)
{
    unsigned long long per = 1ull << 13;
    while (per < kBinRecordsPerBlock && per * 512 < records)
        per <<= 1;
    return per;
}

// records of an accumulation chunk: 2^17, less for renders of few records
static unsigned bin_accum_chunk(unsigned long long records)
{
    unsigned chunk = 1u << 12;
    while (chunk < (1u << 17) && (unsigned long long)chunk * 1024 < records)
        chunk <<= 1;
    return chunk;
}

size_t bin_scratch_hist_words(unsigned long long records, int ntiles)
{
    // (a render of fewer records may take more of its smaller blocks: at
    // most 512 while they are smaller than 2^18)
    const unsigned long long blocks =
        std::max<unsigned long long>(512, (records + kBinRecordsPerBlock - 1) / kBinRecordsPerBlock);
    return (size_t)blocks * (size_t)ntiles;
}

int launch_bin_accumulate(const BinScratch &b, unsigned long long n_records,
                          unsigned long long cells, void *buf, int word_bytes, int r,
                          int real_bytes, hipStream_t s, const unsigned *skip)
{
    const int tile_bits = r > 0 ? kBinTileBitsColour : kBinTileBits;
    const int ntiles = (int)((cells + (1ull << tile_bits) - 1) >> tile_bits);
    if (ntiles > kBinMaxTiles || n_records > 0xFFFFFFFFull || r < 0 || r > 4 ||
        (r > 0 && (real_bytes != 4 && real_bytes != 8)))
        return (int)hipErrorInvalidValue;
    const unsigned long long per = bin_block_records(n_records);
    const unsigned chunk = bin_accum_chunk(n_records);
    const int nblocks = (int)std::max<unsigned long long>(1, (n_records + per - 1) / per);
    const size_t hist_lds = sizeof(unsigned) * (size_t)ntiles;
    hipLaunchKernelGGL(bin_hist_kernel, dim3(nblocks), dim3(kBinBlock), hist_lds, s, b.rec,
                       n_records, per, tile_bits, ntiles, b.hist);
    hipLaunchKernelGGL(bin_colscan_kernel, dim3((ntiles + kScanTiles - 1) / kScanTiles),
                       dim3(kScanTiles * kScanParts), 0, s, b.hist, nblocks, ntiles, b.total);
    unsigned *cstart = b.total + ntiles;
    hipLaunchKernelGGL(bin_tilescan_kernel, dim3(1), dim3(1024), 0, s, b.total, ntiles, chunk,
                       b.start, cstart);
    if (r == 0) {
        if (ntiles <= 4096)
            hipLaunchKernelGGL(bin_scatter_kernel<32>, dim3(nblocks), dim3(kScatterLanes),
                               scatter_lds(ntiles, 32), s, b.rec, n_records, per, tile_bits,
                               ntiles, b.hist, b.start, b.sorted);
        else
            hipLaunchKernelGGL(bin_scatter_kernel<16>, dim3(nblocks), dim3(kScatterLanes),
                               scatter_lds(ntiles, 16), s, b.rec, n_records, per, tile_bits,
                               ntiles, b.hist, b.start, b.sorted);
    } else {
        with_colour_record(r, real_bytes, [&](auto real, auto words) {
            launch_scatter_pay<decltype(real), decltype(words)::value>(b, n_records, per, nblocks,
                                                                       tile_bits, ntiles, r, s);
        });
    }
    // accumulation work items (at most ntiles + n_records / chunk in all)
    const unsigned items = (unsigned)((unsigned long long)ntiles + n_records / chunk);
    if (r == 0) {
        const size_t tile_lds = sizeof(unsigned) << kBinTileBits;
        if (word_bytes == 8)
            hipLaunchKernelGGL((bin_accum_kernel<unsigned long long>), dim3(items), dim3(1024),
                               tile_lds, s, b.sorted, b.start, cstart, ntiles, tile_bits, cells,
                               chunk, skip, (unsigned long long *)buf);
        else
            hipLaunchKernelGGL((bin_accum_kernel<unsigned>), dim3(items), dim3(1024), tile_lds,
                               s, b.sorted, b.start, cstart, ntiles, tile_bits, cells,
                               chunk, skip, (unsigned *)buf);
        return (int)hipGetLastError();
    }
    with_colour_record(r, real_bytes, [&](auto real, auto words) {
        launch_accum_colour<decltype(real), decltype(words)::value>(
            b, items, r, cstart, ntiles, cells, chunk, skip, buf, word_bytes, s);
    });
    return (int)hipGetLastError();
}

int prepare_bin_kernels()
{
    // the accumulate kernel takes a whole tile of counts in LDS (128 KiB)
    const int tile_lds = (int)(sizeof(unsigned) << kBinTileBits);
    hipError_t e = hipFuncSetAttribute((const void *)bin_accum_kernel<unsigned long long>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, tile_lds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)bin_accum_kernel<unsigned>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, tile_lds);
    // the scatter kernel: chunks of 32 records a lane up to 4096 tiles, of
    // 16 up to 8192
    static_assert(scatter_lds(4096, 32) <= 160 * 1024, "scatter chunk beyond the LDS");
    static_assert(accum_colour_lds() <= 160 * 1024, "colour tile beyond the LDS");
    static_assert(scatter_lds(kBinMaxTiles, 16) <= 160 * 1024, "scatter chunk beyond the LDS");
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)bin_scatter_kernel<32>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)scatter_lds(4096, 32));
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)bin_scatter_kernel<16>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)scatter_lds(kBinMaxTiles, 16));
    if (e == hipSuccess)
        e = prepare_colour<float, 4>();
    if (e == hipSuccess)
        e = prepare_colour<float, 8>();
    if (e == hipSuccess)
        e = prepare_colour<double, 8>();
    if (e == hipSuccess)
        e = prepare_colour<double, 12>();
    return (int)e;
}

} // namespace ffr
