// Binning of miss records: the cell updates that miss the walker kernels'
// LDS cell caches, of one flame or of the flames of a batched launch.
//
// Scattered global atomics are resolved at the memory side at about 20 G/s
// on this device, and a missed update of a three-colour cell takes four.
// The 4K colour flame (FP32, 2^32 samples, 3.5 % of them missed) spent 18 of
// 71 ms waiting for them and rendered in 77 to 87 ms; a batch of 24 flames
// (6.5e9 samples, 31 % missed) in 390 ms, the rate of its atomics.  As
// records the misses cost their trips through memory instead: written once
// by the walker, read twice, written once, read once.  The 4K render takes
// 56 ms, of which 4.5 are here, the batch 189 ms, of which 45.
//
// The walkers' waves fill chunks of records, each of one flame.
//   hist     workgroups with a range of the chunks: an LDS histogram over
//            the flame's tiles, added to the tiles' counts where the flame
//            changes
//   scan     the tiles' places in the sorted records, and their
//            accumulation chunks; clears the counts for the next round
//   scatter  stages of a chunk or two of one flame are put into tile order
//            in LDS, each tile's part takes its place with one atomic (a
//            lane per tile: adjacent words), and goes out in whole pieces
//   accum    workgroups take the chunks in turn: counts and colour sums in
//            LDS, then one add per word of each occupied cell
// Per round of 2^28 records of 16 bytes: hist 0.31 ms, scatter 1.26 ms,
// accum 0.77 ms (the scatter moves 8 GB: 6.8 TB/s).  A round costs 0.35 ms
// more, while the walkers' caches are flushed and fill again.
#include "bin_common.hpp"
#include "util_kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace ffr {

namespace {

constexpr int kLanes = 1024;
constexpr unsigned kMissChunk = 1u << 16; // records of an accumulation chunk

// a record as the pieces that move: NW 1 one word, else 16-byte pieces
template <int NW> struct Piece {
    using type = uint4;
    static constexpr int n = NW / 4;
};
template <> struct Piece<1> {
    using type = unsigned;
    static constexpr int n = 1;
};
__device__ __forceinline__ unsigned cell_of(unsigned p) { return p; }
__device__ __forceinline__ unsigned cell_of(uint4 p) { return p.x; }

// no chunk taken, every workgroup's first task; the tiles' counts 0
__global__ void miss_init_kernel(MissCtrl *ctrl, MissPool *pool, int groups,
                                 uint64_t task_walkers, unsigned *count, int tiles)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < groups) {
        ctrl[i].next = (uint64_t)i * task_walkers;
        ctrl[i].resume = 0;
    }
    if (i == 0) {
        pool->next = 0;
        pool->used = 0;
    }
    for (int t = i; t < tiles; t += (int)(gridDim.x * blockDim.x))
        count[t] = 0;
}

// the chunks [k0, k1) of this workgroup
__device__ __forceinline__ void my_chunks(unsigned used, unsigned &k0, unsigned &k1)
{
    const unsigned per = (used + gridDim.x - 1) / gridDim.x;
    k0 = min(used, blockIdx.x * per);
    k1 = min(used, k0 + per);
}

template <int NW>
__global__ void __launch_bounds__(kLanes)
    miss_hist_kernel(const unsigned *rec, const MissChunk *info, const MissPool *pool,
                     unsigned chunks, const MissFlame *flames, int tile_bits, unsigned *count)
{
    constexpr unsigned kChunk = miss_chunk(NW);
    constexpr int kPer = (int)(kChunk / kLanes); // records a lane per chunk
    extern __shared__ unsigned h[];
    unsigned k0, k1;
    my_chunks(min(pool->next, chunks), k0, k1);
    unsigned flame = kNoChunk;
    int tiles = 0, tile0 = 0;
    auto flush = [&]() {
        __syncthreads();
        for (int t = (int)threadIdx.x; t < tiles; t += kLanes)
            if (h[t])
                atomicAdd(&count[tile0 + t], h[t]);
    };
    for (unsigned k = k0; k < k1; ++k) {
        const MissChunk c = info[k];
        if (c.flame != flame) {
            flush();
            flame = c.flame;
            tiles = flames[flame].tiles;
            tile0 = flames[flame].tile0;
            __syncthreads();
            for (int t = (int)threadIdx.x; t < tiles; t += kLanes)
                h[t] = 0;
            __syncthreads();
        }
        const unsigned *from = rec + (size_t)k * kChunk * NW;
        unsigned cell[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const unsigned i = (unsigned)j * kLanes + threadIdx.x;
            cell[j] = from[(size_t)(i < c.n ? i : 0) * NW];
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if ((unsigned)j * kLanes + threadIdx.x < c.n)
                atomicAdd(&h[cell[j] >> tile_bits], 1u);
    }
    flush();
}

// exclusive scans over all tiles (one workgroup): of their records (into
// cursor) and of their accumulation chunks (cstart); start[t + 1] ends tile
// t's records
__global__ void __launch_bounds__(kLanes)
    miss_scan_kernel(unsigned *count, int tiles, unsigned *cursor, unsigned *start,
                     unsigned *cstart, MissPool *pool, unsigned chunks)
{
    __shared__ unsigned part[kLanes], cpart[kLanes];
    const int tid = (int)threadIdx.x;
    const int per = (tiles + kLanes - 1) / kLanes;
    const int t0 = tid * per;
    unsigned s = 0, c = 0;
    for (int k = 0; k < per; ++k)
        if (t0 + k < tiles) {
            const unsigned n = count[t0 + k];
            s += n;
            c += (n + kMissChunk - 1) / kMissChunk;
        }
    part[tid] = s;
    cpart[tid] = c;
    __syncthreads();
    for (int off = 1; off < kLanes; off <<= 1) {
        const unsigned v = tid >= off ? part[tid - off] : 0u;
        const unsigned w = tid >= off ? cpart[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        cpart[tid] += w;
        __syncthreads();
    }
    unsigned run = tid ? part[tid - 1] : 0u, crun = tid ? cpart[tid - 1] : 0u;
    for (int k = 0; k < per; ++k)
        if (t0 + k < tiles) {
            const unsigned n = count[t0 + k];
            count[t0 + k] = 0;
            cursor[t0 + k] = run;
            start[t0 + k] = run;
            cstart[t0 + k] = crun;
            run += n;
            crun += (n + kMissChunk - 1) / kMissChunk;
        }
    if (tid == kLanes - 1) {
        start[tiles] = part[tid];
        cstart[tiles] = cpart[tid];
        pool->used = min(pool->next, chunks);
        pool->next = 0;
    }
}

constexpr size_t miss_scatter_lds(int tiles, int per, int nw)
{
    return sizeof(unsigned) * ((size_t)nw * kLanes * (size_t)per + 2 * (size_t)tiles + 16);
}

template <int PER, int NW>
__global__ void __launch_bounds__(kLanes)
    miss_scatter_kernel(const unsigned *rec, const MissChunk *info, const MissPool *pool,
                        const MissFlame *flames, int tile_bits, int max_tiles, unsigned *cursor,
                        unsigned *sorted)
{
    using P = typename Piece<NW>::type;
    constexpr int NP = Piece<NW>::n;
    constexpr unsigned kChunk = miss_chunk(NW);
    constexpr unsigned kStage = (unsigned)(kLanes * PER);
    constexpr unsigned kParts = kStage >= kChunk ? 1u : kChunk / kStage; // stages of a chunk
    static_assert(kStage <= 2 * kChunk && kChunk % kLanes == 0, "a stage holds one chunk or two");
    extern __shared__ uint4 lds[];
    P *stage = reinterpret_cast<P *>(lds);                                     // [NP][kStage]
    unsigned *cur = reinterpret_cast<unsigned *>(stage + (size_t)NP * kStage); // [tiles] place
    unsigned *off = cur + max_tiles;                                           // [tiles]
    unsigned *wsum = off + max_tiles;                                          // [16]
    const int tid = (int)threadIdx.x;
    P *out = reinterpret_cast<P *>(sorted);
    unsigned k0, k1;
    my_chunks(pool->used, k0, k1);
    // a stage: up to n[0] records at `from`, and n[1] of the next chunk
    struct Stage {
        const P *from;
        unsigned n[2];
        int tiles, tile0;
    };
    unsigned k = k0, part = 0; // the next stage's chunk
    auto next_stage = [&](Stage &g) {
        const MissChunk c = info[k];
        g.tiles = flames[c.flame].tiles;
        g.tile0 = flames[c.flame].tile0;
        g.from = reinterpret_cast<const P *>(rec + ((size_t)k * kChunk + part * kStage) * NW);
        g.n[1] = 0;
        if constexpr (kParts > 1) {
            const unsigned at = part * kStage;
            g.n[0] = c.n > at ? min(c.n - at, kStage) : 0u;
            if (++part == kParts) {
                part = 0;
                ++k;
            }
        } else {
            g.n[0] = c.n;
            ++k;
            if constexpr (kStage > kChunk) {
                if (k < k1) {
                    const MissChunk d = info[k];
                    if (d.flame == c.flame) {
                        g.n[1] = d.n;
                        ++k;
                    }
                }
            }
        }
    };
    // record j of this lane
    auto in = [&](const Stage &g, int j) {
        const unsigned i = (unsigned)j * kLanes + (unsigned)tid;
        return (unsigned)j * kLanes < kChunk ? i < g.n[0] : i - kChunk < g.n[1];
    };
    P v[PER][NP];
    auto load = [&](const Stage &g) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const unsigned i = in(g, j) ? (unsigned)j * kLanes + (unsigned)tid : 0u;
#pragma unroll
            for (int q = 0; q < NP; ++q)
                v[j][q] = g.from[(size_t)i * NP + q];
        }
    };
    if (k == k1)
        return;
    Stage g;
    next_stage(g);
    for (int t = tid; t < g.tiles; t += kLanes)
        off[t] = 0;
    load(g);
    lds_barrier();
    for (;;) {
        // each record's rank in its tile's part of the stage
        unsigned at[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j)
            at[j] = in(g, j) ? atomicAdd(&off[cell_of(v[j][0]) >> tile_bits], 1u) : 0u;
        lds_barrier();
        // the tiles' parts take their places (a lane per tile), while the
        // scan makes their offsets in the stage
        for (int t = tid; t < g.tiles; t += kLanes) {
            const unsigned n = off[t];
            cur[t] = n ? atomicAdd(&cursor[g.tile0 + t], n) : 0u;
        }
        lds_barrier();
        const unsigned total = lds_scan(off, g.tiles, wsum);
        lds_barrier();
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (in(g, j)) {
                const unsigned pos = off[cell_of(v[j][0]) >> tile_bits] + at[j];
#pragma unroll
                for (int q = 0; q < NP; ++q)
                    stage[(size_t)q * kStage + pos] = v[j][q];
            }
        const bool more = k < k1;
        if (more) {
            next_stage(g);
            load(g);
        }
        lds_barrier();
        for (unsigned i = (unsigned)tid; i < total; i += kLanes) {
            const P first = stage[i];
            const unsigned t = cell_of(first) >> tile_bits;
            P *dst = out + (size_t)(cur[t] + (i - off[t])) * NP;
            dst[0] = first;
#pragma unroll
            for (int q = 1; q < NP; ++q)
                dst[q] = stage[(size_t)q * kStage + i];
        }
        if (!more)
            break;
        lds_barrier();
        for (int t = tid; t < g.tiles; t += kLanes)
            off[t] = 0;
        lds_barrier();
    }
}

// one accumulation chunk after another: tile t of flame f
template <typename CT>
__global__ void __launch_bounds__(kLanes)
    miss_accum_kernel(const unsigned *sorted, const unsigned *start, const unsigned *cstart,
                      int tiles, const unsigned *tile_flame, const MissFlame *flames)
{
    constexpr unsigned kTile = 1u << kBinTileBits;
    extern __shared__ unsigned cnt[];
    const unsigned items = cstart[tiles];
    for (unsigned w = blockIdx.x; w < items; w += gridDim.x) {
        const int t = last_not_above(cstart, tiles, w);
        const MissFlame f = flames[tile_flame[t]];
        const bool shared = cstart[t + 1] - cstart[t] > 1;
        const unsigned s0 = start[t] + (w - cstart[t]) * kMissChunk;
        const unsigned s1 = min(start[t + 1], s0 + kMissChunk);
        const unsigned long long c0 = (unsigned long long)(t - f.tile0) * kTile;
        const unsigned ncell = (unsigned)min((unsigned long long)kTile, f.cells - c0);
        for (unsigned i = threadIdx.x; i < ((ncell + 31u) & ~31u); i += kLanes)
            cnt[i] = 0;
        __syncthreads();
        for (unsigned i0 = s0 + threadIdx.x; i0 < s1; i0 += kLanes * 8) {
            unsigned k[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned i = i0 + (unsigned)j * kLanes;
                k[j] = sorted[i < s1 ? i : i0];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (i0 + (unsigned)j * kLanes < s1)
                    atomicAdd(&cnt[tile_word(k[j] & (kTile - 1u))], 1u);
        }
        __syncthreads();
        CT *buf = static_cast<CT *>(f.buf) + c0;
        for (unsigned i = threadIdx.x; i < ncell; i += kLanes) {
            const unsigned n = cnt[tile_word(i)];
            if (!n)
                continue;
            if (shared)
                atomicAdd(&buf[i], (CT)n);
            else
                buf[i] += (CT)n;
        }
        __syncthreads();
    }
}

constexpr int kColourTile = 1 << kBinTileBitsColour;

// 8-byte words: u64 counts and f64 colour sums
template <typename PR, int NW>
__global__ void __launch_bounds__(kLanes)
    miss_accum_colour_kernel(const uint4 *sorted, const unsigned *start, const unsigned *cstart,
                             int tiles, const unsigned *tile_flame, const MissFlame *flames)
{
    constexpr int kReal = (int)sizeof(PR) / 4;
    constexpr int NR = (NW - 1) / kReal < 4 ? (NW - 1) / kReal : 4;
    constexpr int kUnroll = 4;
    extern __shared__ unsigned long long lds64[];
    double *col = reinterpret_cast<double *>(lds64);                     // [NR][kColourTile]
    unsigned *cnt = reinterpret_cast<unsigned *>(col + 4 * kColourTile); // [kColourTile]
    const unsigned items = cstart[tiles];
    for (unsigned w = blockIdx.x; w < items; w += gridDim.x) {
        const int t = last_not_above(cstart, tiles, w);
        const MissFlame f = flames[tile_flame[t]];
        const int nr = f.r;
        const bool shared = cstart[t + 1] - cstart[t] > 1;
        const unsigned s0 = start[t] + (w - cstart[t]) * kMissChunk;
        const unsigned s1 = min(start[t + 1], s0 + kMissChunk);
        const unsigned long long c0 = (unsigned long long)(t - f.tile0) * kColourTile;
        const unsigned ncell = (unsigned)min((unsigned long long)kColourTile, f.cells - c0);
        for (unsigned i = threadIdx.x; i < ((ncell + 31u) & ~31u); i += kLanes) {
            cnt[i] = 0;
            for (int j = 0; j < nr; ++j)
                col[j * kColourTile + i] = 0.0;
        }
        __syncthreads();
        for (unsigned i0 = s0 + threadIdx.x; i0 < s1; i0 += kLanes * kUnroll) {
            unsigned v[kUnroll][NW];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const unsigned i = i0 + (unsigned)u * kLanes;
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
            for (int u = 0; u < kUnroll; ++u) {
                if (i0 + (unsigned)u * kLanes >= s1)
                    break;
                const unsigned cw = tile_word(v[u][0] & (kColourTile - 1));
                atomicAdd(&cnt[cw], 1u);
#pragma unroll
                for (int j = 0; j < NR; ++j)
                    if (j < nr)
                        atomicAdd(&col[j * kColourTile + cw],
                                  get_real<PR>(&v[u][1 + j * kReal]));
            }
        }
        __syncthreads();
        const int words = 1 + nr;
        for (unsigned i = threadIdx.x; i < ncell; i += kLanes) {
            const unsigned cw = tile_word(i);
            const unsigned n = cnt[cw];
            if (!n)
                continue;
            unsigned long long *cell = static_cast<unsigned long long *>(f.buf) +
                                       (c0 + i) * (unsigned long long)words;
            double *colour = reinterpret_cast<double *>(cell + 1);
            if (shared) {
                atomicAdd(cell, (unsigned long long)n);
                for (int j = 0; j < nr; ++j)
                    unsafeAtomicAdd(&colour[j], col[j * kColourTile + cw]);
            } else {
                *cell += (unsigned long long)n;
                for (int j = 0; j < nr; ++j)
                    colour[j] += col[j * kColourTile + cw];
            }
        }
        __syncthreads();
    }
}

constexpr size_t accum_colour_lds()
{
    return sizeof(double) * 4 * kColourTile + sizeof(unsigned) * kColourTile;
}

// the scatter's records a lane per chunk, by record words and tiles: what
// the LDS holds
constexpr int kScatterTiles = 3072;
constexpr int scatter_per(int nw, bool many)
{
    return nw == 1 ? (many ? 16 : 32) : nw == 4 ? (many ? 4 : 8) : nw == 8 ? (many ? 2 : 4) : (many ? 1 : 2);
}

// f(walker real, record words) for a record size
template <typename F> void with_record(int words, int real_bytes, F &&f)
{
    if (words == 1)
        f(float(), std::integral_constant<int, 1>());
    else if (real_bytes == 8 && words == 8)
        f(double(), std::integral_constant<int, 8>());
    else if (real_bytes == 8)
        f(double(), std::integral_constant<int, 12>());
    else if (words == 4)
        f(float(), std::integral_constant<int, 4>());
    else
        f(float(), std::integral_constant<int, 8>());
}

template <int NW> hipError_t prepare_scatter()
{
    static_assert(miss_scatter_lds(kScatterTiles, scatter_per(NW, false), NW) <= 160 * 1024, "scatter chunk beyond the LDS");
    static_assert(miss_scatter_lds(kBinMaxTiles, scatter_per(NW, true), NW) <= 160 * 1024, "scatter chunk beyond the LDS");
    hipError_t e = hipFuncSetAttribute(
        (const void *)miss_scatter_kernel<scatter_per(NW, false), NW>,
        hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)miss_scatter_lds(kScatterTiles, scatter_per(NW, false), NW));
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)miss_scatter_kernel<scatter_per(NW, true), NW>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)miss_scatter_lds(kBinMaxTiles, scatter_per(NW, true), NW));
    return e;
}

} // namespace

int launch_miss_init(const MissScratch &x, uint64_t task_walkers, hipStream_t s)
{
    const int n = std::max(x.groups, x.tiles);
    hipLaunchKernelGGL(miss_init_kernel, dim3((n + 255) / 256), dim3(256), 0, s, x.ctrl, x.pool,
                       x.groups, task_walkers, x.count, x.tiles);
    return (int)hipGetLastError();
}

int launch_miss_round(const MissScratch &x, int word_bytes, hipStream_t s)
{
    const int tile_bits = x.words == 1 ? kBinTileBits : kBinTileBitsColour;
    if (x.max_tiles > kBinMaxTiles || x.max_tiles <= 0 || x.groups <= 0 ||
        (x.words > 1 && word_bytes != 8))
        return (int)hipErrorInvalidValue;
    const bool many = x.max_tiles > kScatterTiles;
    with_record(x.words, x.real_bytes, [&](auto real, auto words) {
        constexpr int NW = decltype(words)::value;
        hipLaunchKernelGGL((miss_hist_kernel<NW>), dim3(2 * x.cu_count), dim3(kLanes),
                           sizeof(unsigned) * (size_t)x.max_tiles, s, x.rec, x.info, x.pool,
                           x.chunks, x.flames, tile_bits, x.count);
        hipLaunchKernelGGL(miss_scan_kernel, dim3(1), dim3(kLanes), 0, s, x.count, x.tiles,
                           x.cursor, x.start, x.cstart, x.pool, x.chunks);
        auto scatter = [&](auto kern, int per) {
            hipLaunchKernelGGL(kern, dim3(x.cu_count), dim3(kLanes),
                               miss_scatter_lds(x.max_tiles, per, NW), s, x.rec, x.info, x.pool,
                               x.flames, tile_bits, x.max_tiles, x.cursor, x.sorted);
        };
        if (many)
            scatter(miss_scatter_kernel<scatter_per(NW, true), NW>, scatter_per(NW, true));
        else
            scatter(miss_scatter_kernel<scatter_per(NW, false), NW>, scatter_per(NW, false));
        // (the tiles' LDS leaves one workgroup per CU)
        if constexpr (NW == 1) {
            const size_t lds = sizeof(unsigned) << kBinTileBits;
            if (word_bytes == 8)
                hipLaunchKernelGGL((miss_accum_kernel<unsigned long long>), dim3(x.cu_count),
                                   dim3(kLanes), lds, s, x.sorted, x.start, x.cstart, x.tiles,
                                   x.tile_flame, x.flames);
            else
                hipLaunchKernelGGL((miss_accum_kernel<unsigned>), dim3(x.cu_count), dim3(kLanes),
                                   lds, s, x.sorted, x.start, x.cstart, x.tiles, x.tile_flame,
                                   x.flames);
        } else {
            hipLaunchKernelGGL((miss_accum_colour_kernel<decltype(real), NW>), dim3(x.cu_count),
                               dim3(kLanes), accum_colour_lds(), s, (const uint4 *)x.sorted,
                               x.start, x.cstart, x.tiles, x.tile_flame, x.flames);
        }
    });
    return (int)hipGetLastError();
}

int prepare_miss_kernels()
{
    auto limit = [](const void *k, size_t bytes) {
        return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    };
    hipError_t e = prepare_scatter<1>();
    if (e == hipSuccess)
        e = prepare_scatter<4>();
    if (e == hipSuccess)
        e = prepare_scatter<8>();
    if (e == hipSuccess)
        e = prepare_scatter<12>();
    const void *counts[] = {(const void *)miss_accum_kernel<unsigned long long>,
                            (const void *)miss_accum_kernel<unsigned>};
    for (const void *k : counts)
        if (e == hipSuccess)
            e = limit(k, sizeof(unsigned) << kBinTileBits);
    const void *colours[] = {(const void *)miss_accum_colour_kernel<float, 4>,
                             (const void *)miss_accum_colour_kernel<float, 8>,
                             (const void *)miss_accum_colour_kernel<double, 8>,
                             (const void *)miss_accum_colour_kernel<double, 12>};
    for (const void *k : colours)
        if (e == hipSuccess)
            e = limit(k, accum_colour_lds());
    return (int)e;
}

} // namespace ffr
