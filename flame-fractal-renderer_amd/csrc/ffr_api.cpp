// C ABI of the renderer (include/ffr.h): flame parsing, device buffers,
// kernel launches and statistics.
#include "../../include/ffr.h"

#include "flame_model.hpp"
#include "rtc.hpp"
#include "util_kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <deque>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <memory>
#include <system_error>
#include <type_traits>
#include <string>
#include <vector>

using namespace ffr;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
    g_err = msg;
    return code;
}

#define HIP_TRY(call)                                                                  \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess)                                                          \
            return fail(FFR_E_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Colour flames switch to binned accumulation after a render of at least
// kBinColourMinSamples samples whose updates past the LDS cache (a count and
// each colour word) reached so many words per sample.  Where those are miss
// records: 2^30 samples of 68 batch flames of 2048^2 cells with three
// colours, and five of them up to 5700^2, take 0.55-0.65 of the binned time
// at 0.5-0.7 words, 0.71-0.80 (FP32) and 0.81-0.94 (FP64) at 1.1-1.5,
// 0.86-0.92 and 0.97-1.07 at 2.0, 0.96-1.01 and 1.13-1.16 at 2.7-3.0.  Where
// they are atomics (4-byte words): binned renders faster from 0.55-0.6 words
// on (1.03-1.42x at 0.6-0.9, 2-4x from 1.1 on), slower below 0.5.
constexpr uint64_t kBinColourMinSamples = 1ull << 26;
constexpr double kBinColourRecords = 1.9;
constexpr double kBinColourAtomics = 0.6;

// the kernels take the xform record offsets as constants (XformLay<D>);
// the table builder must lay records out the same way
template <int D> bool layout_matches(const XformLayout &l)
{
    using K = XformLay<D>;
    return l.preA == K::preA && l.preb == K::preb && l.postA == K::postA &&
           l.postb == K::postb && l.speed == K::speed && l.has_color == K::has_color &&
           l.has_pre == K::has_pre && l.has_post == K::has_post && l.color == K::color;
}
bool layout_matches_kernels(const XformLayout &l, int dims)
{
    return dims == 1 ? layout_matches<1>(l) : dims == 2 ? layout_matches<2>(l)
                                             : dims == 3 && layout_matches<3>(l);
}

struct DevTables {
    void *table = nullptr;
    unsigned long long *masks = nullptr;
    size_t table_bytes = 0;
    int tab_reals = 0;
};

bool free_idle_records(); // (of the current device, below)

// device memory that a call cannot do without: idle record memory makes way
template <typename T> hipError_t device_malloc(T **p, size_t bytes)
{
    hipError_t e = hipMalloc((void **)p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        if (free_idle_records())
            e = hipMalloc((void **)p, bytes);
    }
    return e;
}

// grow a device allocation to at least `bytes` (contents not kept)
hipError_t ensure_device(void **p, size_t &have, size_t bytes)
{
    if (have >= bytes)
        return hipSuccess;
    (void)hipFree(*p);
    *p = nullptr;
    have = 0;
    hipError_t e = device_malloc(p, bytes);
    if (e == hipSuccess)
        have = bytes;
    return e;
}

} // namespace

// Miss records: the memory of a render's launches (or of a batch's kinds,
// which run one after another)
struct MissMemory {
    void *rec = nullptr, *sorted = nullptr, *info = nullptr, *ctrl = nullptr, *state = nullptr;
    size_t rec_bytes = 0, sorted_bytes = 0, info_bytes = 0, ctrl_bytes = 0, state_bytes = 0;

    hipError_t ensure(int groups, int lanes, unsigned chunks, int words, int real_bytes)
    {
        const size_t n = (size_t)chunks * miss_chunk(words) * (size_t)words * 4;
        const size_t pause = real_bytes == 8 ? sizeof(WalkerPause<double>)
                                             : sizeof(WalkerPause<float>);
        hipError_t e = ensure_device(&rec, rec_bytes, n);
        if (e == hipSuccess)
            e = ensure_device(&sorted, sorted_bytes, n);
        if (e == hipSuccess)
            e = ensure_device(&info, info_bytes, (size_t)chunks * sizeof(MissChunk));
        if (e == hipSuccess) // (the pool's counters in front)
            e = ensure_device(&ctrl, ctrl_bytes,
                              sizeof(MissCtrl) + (size_t)groups * sizeof(MissCtrl));
        if (e == hipSuccess)
            e = ensure_device(&state, state_bytes, (size_t)groups * (size_t)lanes * pause);
        return e;
    }
    void free_all()
    {
        for (void *p : {rec, sorted, info, ctrl, state})
            (void)hipFree(p);
        *this = MissMemory();
    }
    size_t bytes() const
    {
        return rec_bytes + sorted_bytes + info_bytes + ctrl_bytes + state_bytes;
    }
};

// The scratch of binned accumulation: of a renderer's binned renders, or of a
// split one's
struct BinMemory {
    BinScratch b;
    size_t rec = 0, sorted = 0, hist = 0, total = 0, start = 0, pay = 0, pay_sorted = 0; // bytes

    // what the arrays take for `cap` records of ncol colours
    static BinMemory sizes(uint64_t cells, int ncol, uint64_t cap, int real_bytes)
    {
        const int tile_bits = ncol > 0 ? kBinTileBitsColour : kBinTileBits;
        const size_t ntiles = (size_t)((cells + (1ull << tile_bits) - 1) >> tile_bits);
        BinMemory n;
        n.rec = (size_t)cap * 4;
        n.hist = bin_scratch_hist_words(cap, (int)ntiles) * 4;
        // per tile: records, then the first accumulation work item; the regions
        n.total = n.start = 2 * (ntiles + 1) * 4;
        if (ncol == 0) {
            n.sorted = n.rec;
        } else {
            // the records' colours, component i at i * capacity, and the
            // whole records in tile order
            n.pay = (size_t)ncol * (size_t)cap * (size_t)real_bytes;
            n.pay_sorted = (size_t)cap * (size_t)(4 * record_words(ncol, real_bytes));
        }
        return n;
    }
    size_t bytes() const { return rec + sorted + hist + total + start + pay + pay_sorted; }
    // the bytes that ensure(n) would allocate
    size_t growth(const BinMemory &n) const
    {
        auto more = [](size_t have, size_t need) { return need > have ? need : 0; };
        return more(rec, n.rec) + more(sorted, n.sorted) + more(hist, n.hist) +
               more(total, n.total) + more(start, n.start) + more(pay, n.pay) +
               more(pay_sorted, n.pay_sorted);
    }
    // grown as needed
    hipError_t ensure(const BinMemory &n, uint64_t cap)
    {
        b.capacity = 0;
        hipError_t e = ensure_device((void **)&b.rec, rec, n.rec);
        if (e == hipSuccess)
            e = ensure_device((void **)&b.sorted, sorted, n.sorted);
        if (e == hipSuccess)
            e = ensure_device((void **)&b.hist, hist, n.hist);
        if (e == hipSuccess)
            e = ensure_device((void **)&b.total, total, n.total);
        if (e == hipSuccess)
            e = ensure_device((void **)&b.start, start, n.start);
        if (e == hipSuccess)
            e = ensure_device(&b.pay, pay, n.pay);
        if (e == hipSuccess)
            e = ensure_device(&b.pay_sorted, pay_sorted, n.pay_sorted);
        if (e == hipSuccess)
            b.capacity = cap;
        return e;
    }
    void free_all()
    {
        for (void *p : {(void *)b.rec, (void *)b.sorted, (void *)b.hist, (void *)b.total,
                        (void *)b.start, b.pay, b.pay_sorted})
            (void)hipFree(p);
        *this = BinMemory();
    }
};

// Record memory that a render (or a batch's pass) can do without, lent for
// the time from its launch to the wait for it.  A device's renderers share
// what lies idle, and it makes way for any other allocation of the library
// (device_malloc).  One idle memory outlives the last of them (kKeepBytes):
// the driver wipes freed memory in the background, and a program that makes
// a renderer per flame, frees gigabytes with each and has gone through the
// device's memory once waits 0.1 to 1 s in an allocation for that.
struct RecordMemory {
    MissMemory miss;
    BinMemory split; // split walkers
    ~RecordMemory()
    {
        miss.free_all();
        split.free_all();
    }
    size_t bytes() const { return miss.bytes() + split.bytes(); }
};

struct RecordPool {
    // idle memories kept while there are renderers, the last one whatever its
    // size (several for programs that render on several threads)
    static constexpr size_t kIdle = 4, kIdleBytes = (size_t)16 << 30;
    // the largest that is kept after them (miss records take 8 GiB)
    static constexpr size_t kKeepBytes = (size_t)10 << 30;
    using Idle = std::vector<std::unique_ptr<RecordMemory>>; // oldest first
    std::mutex lock;
    Idle idle;

    // a device's, for the life of the process
    static RecordPool *of_device(int device)
    {
        static std::mutex *m = new std::mutex;
        static std::map<int, RecordPool *> *pools = new std::map<int, RecordPool *>;
        std::lock_guard<std::mutex> g(*m);
        RecordPool *&p = (*pools)[device];
        if (!p)
            p = new RecordPool;
        return p;
    }
    std::unique_ptr<RecordMemory> take()
    {
        std::lock_guard<std::mutex> g(lock);
        if (idle.empty())
            return std::make_unique<RecordMemory>();
        std::unique_ptr<RecordMemory> m = std::move(idle.back());
        idle.pop_back();
        return m;
    }
    void give(std::unique_ptr<RecordMemory> m)
    {
        Idle out; // (freed outside the lock)
        std::lock_guard<std::mutex> g(lock);
        size_t bytes = m->bytes();
        for (const auto &i : idle)
            bytes += i->bytes();
        idle.push_back(std::move(m));
        while (idle.size() > 1 && (idle.size() > kIdle || bytes > kIdleBytes)) {
            bytes -= idle.front()->bytes();
            out.push_back(std::move(idle.front()));
            idle.erase(idle.begin());
        }
    }
    // the last renderer, batch and server are gone
    void rest()
    {
        Idle out;
        std::lock_guard<std::mutex> g(lock);
        out.swap(idle);
        if (!out.empty() && out.back()->bytes() <= kKeepBytes) {
            idle.push_back(std::move(out.back()));
            out.pop_back();
        }
    }
    bool free_idle()
    {
        Idle out;
        std::lock_guard<std::mutex> g(lock);
        out.swap(idle);
        return !out.empty();
    }
};

// a renderer's (or a batch's) loan
struct RecordLoan {
    // held by every renderer and batch of a device
    struct Users {
        RecordPool *pool;
        ~Users() { pool->rest(); }
    };
    std::shared_ptr<Users> users;
    std::unique_ptr<RecordMemory> mem;

    void open(int device)
    {
        static std::mutex *m = new std::mutex;
        static std::map<int, std::weak_ptr<Users>> *all = new std::map<int, std::weak_ptr<Users>>;
        std::lock_guard<std::mutex> g(*m);
        users = (*all)[device].lock();
        if (!users) {
            users.reset(new Users{RecordPool::of_device(device)});
            (*all)[device] = users;
        }
    }
    RecordMemory &get()
    {
        if (!mem)
            mem = users->pool->take();
        return *mem;
    }
    // (nothing that uses the memory runs any more)
    void give_back()
    {
        if (mem)
            users->pool->give(std::move(mem));
    }
};

namespace {

bool free_idle_records()
{
    int device = 0;
    return hipGetDevice(&device) == hipSuccess && RecordPool::of_device(device)->free_idle();
}

} // namespace

// The tiles of the flames of a launch with miss records
struct MissTiles {
    void *words = nullptr, *flames = nullptr;
    size_t words_bytes = 0, flames_bytes = 0;
    int tiles = 0, max_tiles = 0;
    // host copies, alive until the device's ones were made
    std::vector<unsigned> tile_flame;
    std::vector<MissFlame> list;

    // flames (buf, cells, r filled in) in tiles of 2^tile_bits cells
    hipError_t set(const std::vector<MissFlame> &fl, int tile_bits, hipStream_t s)
    {
        auto same = [](const MissFlame &x, const MissFlame &y) {
            return x.buf == y.buf && x.cells == y.cells && x.r == y.r;
        };
        if (tiles && fl.size() == list.size() &&
            std::equal(fl.begin(), fl.end(), list.begin(), same))
            return hipSuccess; // (the device has them)
        // copies of the last call may still read the vectors
        hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess)
            return e;
        list = fl;
        tile_flame.clear();
        max_tiles = 0;
        for (size_t i = 0; i < list.size(); ++i) {
            MissFlame &f = list[i];
            f.tile0 = (int)tile_flame.size();
            f.tiles = (int)((f.cells + (1ull << tile_bits) - 1) >> tile_bits);
            max_tiles = std::max(max_tiles, f.tiles);
            tile_flame.insert(tile_flame.end(), (size_t)f.tiles, (unsigned)i);
        }
        const int n = (int)tile_flame.size();
        tiles = 0;
        e = ensure_device(&words, words_bytes, ((size_t)n * 5 + 2) * 4);
        if (e == hipSuccess)
            e = ensure_device(&flames, flames_bytes, list.size() * sizeof(MissFlame));
        if (e == hipSuccess)
            e = hipMemcpyAsync((unsigned *)words + (size_t)n * 4 + 2, tile_flame.data(),
                               (size_t)n * 4, hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(flames, list.data(), list.size() * sizeof(MissFlame),
                               hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            tiles = n;
        return e;
    }
    void free_all()
    {
        (void)hipFree(words);
        (void)hipFree(flames);
        *this = MissTiles();
    }
};

// The rounds (walker launch, then its records binned) of a render, the chunks
// of its records, and the chunk from which its workgroups pause.  Where
// every sample's record fits, one round is enough; else as many as the
// expected misses (rate) fill and two more, and a last launch finishes with
// atomics what is left then.
struct MissRounds {
    unsigned chunks = 0, limit = 0;
    int rounds = 0;
    bool last = false;
};

// The record memory (as much again holds the sorted records): at most an
// eighth of the free memory in all.  The batch of 24 flames (32 GB of records)
// took 216 ms with 1 GB, 195 with 2, 189 with 4 and 185 with 8; the 4K
// colour flame (2.4 GB) 57.7, 56.7 and 55.9 ms with 1, 2 and 4
constexpr size_t kMissBytes = (size_t)4 << 30;
// Renders keep their atomics where the walkers hide them.  While the launch
// fills the device's lanes, by missed words a sample (as atomics miss), 2^28
// to 2^32 samples of 40 flames, atomics over records in time:
//   FP32  0.85-0.96 below 0.09; 0.91-1.06 and once 1.6 at 0.09-0.125; 0.9-1.3
//         at 0.13-0.135 (the 4K colour flame 1.04-1.28, compiled 1.43);
//         1.05-1.8 at 0.16-0.25, 1.2-2.4 at 0.25-0.45
//   FP64  (longer iterations hide more) 0.87-0.95 below 0.28, 0.97-1.02 at
//         0.3, 1.15-1.25 at 0.34 (once 0.85), 1.1-1.4 at 0.43-0.48
// A launch of fewer walkers than lanes takes as long as a full one and misses
// less in it, so the line rises as the walkers fall: 2^27 samples in FP32
// (half the lanes) cross at 0.3, 2^26 between 0.86 (0.96) and 2.4 (2.4), 2^24
// (a sixteenth) below 2.4 (1.28); FP64 2^26 (half) between 0.84 (0.87) and
// 2.4 (2.1).  A batch's flames hide each other's: 64 of them in FP64, 0.61
// words in the mean, 766 / 807 ms.  A first render, which knows no rate, is
// taken to miss 0.6 words: first renders of 86 flames, half of which miss
// under 0.02 and a fifth over 0.44, take with atomics and with records in all
//   FP32  2^25 samples 305 / 313 ms, 2^26 336 / 323, 2^27 428 / 344
//   FP64  2^25 323 / 334, 2^26 357 / 349, 2^27 453 / 387
// (one by one 0.5 to 3.7 times).
constexpr uint64_t kMissMinSamples = 1ull << 24;
constexpr double kMissWords32 = 0.13, kMissWords64 = 0.3, kMissWordsBatch64 = 0.75;
constexpr double kMissWordsUnknown = 0.6;

// rate: the share of the samples that missed (negative: unknown)
static bool miss_worth(double rate, int cell_words, int real_bytes, bool batch,
                       uint64_t walkers, uint64_t lanes)
{
    const double least =
        real_bytes == 4 ? kMissWords32 : batch && rate >= 0 ? kMissWordsBatch64 : kMissWords64;
    const double words = rate < 0 ? kMissWordsUnknown : rate * cell_words;
    return words >= least * std::max(1.0, (double)lanes / (double)std::max<uint64_t>(walkers, 1));
}

static MissRounds miss_rounds(const MissMemory &mem, uint64_t samples, uint64_t tasks, int groups,
                              int lanes, int words, double rate)
{
    const uint64_t chunk = miss_chunk(words), chunk_bytes = chunk * (uint64_t)words * 4;
    const uint64_t waves = ((uint64_t)lanes + 63) / 64;
    // (a wave begins a chunk in each task; a launch whose chunks were used up
    // would leave walkers paused)
    const uint64_t all = miss_chunks_most(samples, (tasks + (uint64_t)groups) * waves, words);
    uint64_t bytes = kMissBytes;
    if (const char *e = std::getenv("FFR_MISS_BYTES"))
        bytes = std::max<uint64_t>((uint64_t)std::atoll(e), 2 * chunk_bytes);
    else if (mem.rec_bytes < std::min(bytes, all * chunk_bytes)) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess)
            return MissRounds();
        bytes = std::max<uint64_t>(mem.rec_bytes, std::min<uint64_t>(bytes, free_b / 16));
    }
    MissRounds m;
    const uint64_t most = bytes / chunk_bytes;
    if (all <= most) {
        m.chunks = m.limit = (unsigned)all;
        m.rounds = 1;
        return m;
    }
    // (the next render may miss somewhat more)
    rate = rate < 0 ? 0.75 : std::min(1.0, 0.02 + 1.3 * rate);
    const uint64_t spare = std::min<uint64_t>(most / 2, (uint64_t)groups * waves);
    m.chunks = (unsigned)most;
    m.limit = (unsigned)(most - spare);
    const double expect = (double)samples * rate / (double)chunk +
                          0.5 * (double)tasks * (double)waves;
    m.rounds = most ? (int)std::min(expect / ((double)m.limit - 0.25 * (double)spare) + 2.0, 4096.0)
                    : 0;
    m.last = true;
    return m;
}

static MissScratch miss_scratch(const MissMemory &m, const MissTiles &t, unsigned chunks,
                                int groups, int words, int real_bytes, int cu_count)
{
    MissScratch x;
    x.rec = (unsigned *)m.rec;
    x.sorted = (unsigned *)m.sorted;
    x.info = (MissChunk *)m.info;
    x.pool = (MissPool *)m.ctrl;
    x.ctrl = (MissCtrl *)m.ctrl + 1;
    x.state = m.state;
    unsigned *w = (unsigned *)t.words;
    x.count = w;
    x.cursor = w + t.tiles;
    x.start = w + 2 * (size_t)t.tiles;
    x.cstart = w + 3 * (size_t)t.tiles + 1;
    x.tile_flame = w + 4 * (size_t)t.tiles + 2;
    x.flames = (MissFlame *)t.flames;
    x.chunks = chunks;
    x.groups = groups;
    x.words = words;
    x.real_bytes = real_bytes;
    x.tiles = t.tiles;
    x.max_tiles = t.max_tiles;
    x.cu_count = cu_count;
    return x;
}

static MissArgs miss_args(const MissScratch &x, unsigned limit)
{
    return MissArgs{x.rec, x.info, x.pool, x.ctrl, x.state, x.chunks, limit};
}

static int prepare_miss_once()
{
    static std::once_flag once;
    static int rc = 0;
    std::call_once(once, [] { rc = prepare_miss_kernels(); });
    return rc;
}

// Pinned chunks through which large host copies go.  The runtime's own copy
// of pageable memory stages through one thread, whose memcpy (and the page
// faults of a new destination) bound it: adding a buffer of 66 MB to another
// and reading it took 7.5 to 9.1 ms.  Here several threads copy chunks while
// the link moves others: 1.9 ms for 66 MB either way (8 threads of 2 MB
// chunks; 2.3 with 6 or 12 of 1 MB, 3.2 of 0.5 MB).  One per device, shared by its
// renderers and given back with the last of them; a copy that finds it in
// use takes the runtime's.  By size, the runtime's copy against this one
// (ms): reads 0.46 / 0.37 of 8 MiB, 0.9-1.3 / 0.6 of 16, 3.1 / 1.2 of 32, 4.8
// / 1.5 of 48; writes 0.24 / 0.33, 0.45 / 0.54, 0.98 / 0.94, 1.7 / 1.4.  The
// first copy also pays 1 to 2.5 ms for the pinned memory, so it is made
// for a copy that wins them back, or once earlier ones would have.  Memory
// that the caller pinned takes the link by itself (0.16 / 0.36 ms of 8 MiB,
// 2.3 / 3.4 of 128).
struct HostStage {
    static constexpr int kThreads = 8, kSlots = 2;
    static constexpr size_t kChunk = (size_t)2 << 20;
    static constexpr size_t kReadBytes = (size_t)8 << 20;
    static constexpr size_t kWriteBytes = (size_t)48 << 20;
    // bytes of copies beyond kReadBytes each from which on it is made
    static constexpr size_t kFirstBytes = (size_t)40 << 20;
    std::mutex busy;
    bool ready = false;
    size_t asked = 0; // bytes of the copies so far beyond kReadBytes each
    char *pin = nullptr;
    hipEvent_t ev[kThreads * kSlots] = {};

    static std::shared_ptr<HostStage> of_device(int device)
    {
        static std::mutex lock;
        static std::map<int, std::weak_ptr<HostStage>> stages;
        std::lock_guard<std::mutex> g(lock);
        std::shared_ptr<HostStage> p = stages[device].lock();
        if (!p) {
            p = std::make_shared<HostStage>();
            stages[device] = p;
        }
        return p;
    }
    // made, or worth it with this copy
    bool wanted(size_t bytes)
    {
        if (!ready)
            asked += bytes - kReadBytes;
        return ready || asked >= kFirstBytes;
    }
    hipError_t init()
    {
        if (ready)
            return hipSuccess;
        hipError_t e = pin ? hipSuccess
                           : hipHostMalloc((void **)&pin, kThreads * kSlots * kChunk,
                                           hipHostMallocDefault);
        for (hipEvent_t &v : ev)
            if (e == hipSuccess && !v)
                e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
        ready = e == hipSuccess;
        return e;
    }
    ~HostStage()
    {
        for (hipEvent_t v : ev)
            if (v)
                (void)hipEventDestroy(v);
        if (pin)
            (void)hipHostFree(pin);
    }
    // host <-> device in stream order; complete on return
    hipError_t copy(int device, hipStream_t s, void *host, void *dev, size_t bytes, bool to_host)
    {
        const size_t n = (bytes + kChunk - 1) / kChunk;
        std::atomic<size_t> next{0};
        std::atomic<int> error{0};
        auto work = [&](int t) {
            hipError_t e = hipSetDevice(device);
            size_t at[kSlots];
            bool used[kSlots] = {};
            auto finish = [&](int k) { // slot k's copy has ended; its chunk to the host
                if (!used[k])
                    return;
                used[k] = false;
                const hipError_t w = hipEventSynchronize(ev[t * kSlots + k]);
                if (e == hipSuccess)
                    e = w;
                if (to_host && e == hipSuccess)
                    std::memcpy((char *)host + at[k], pin + (size_t)(t * kSlots + k) * kChunk,
                                std::min(kChunk, bytes - at[k]));
            };
            int k = 0;
            for (; e == hipSuccess && !error.load(); k = (k + 1) % kSlots) {
                finish(k);
                const size_t i = next.fetch_add(1);
                if (i >= n || e != hipSuccess)
                    break;
                at[k] = i * kChunk;
                const size_t len = std::min(kChunk, bytes - at[k]);
                char *slot = pin + (size_t)(t * kSlots + k) * kChunk;
                if (to_host) {
                    e = hipMemcpyAsync(slot, (char *)dev + at[k], len, hipMemcpyDeviceToHost, s);
                } else {
                    std::memcpy(slot, (char *)host + at[k], len);
                    e = hipMemcpyAsync((char *)dev + at[k], slot, len, hipMemcpyHostToDevice, s);
                }
                if (e == hipSuccess)
                    e = hipEventRecord(ev[t * kSlots + k], s);
                used[k] = e == hipSuccess;
            }
            for (int j = 0; j < kSlots; ++j)
                finish((k + j) % kSlots);
            if (e != hipSuccess)
                error = (int)e;
        };
        std::thread threads[kThreads - 1];
        try {
            for (int t = 1; t < kThreads; ++t)
                threads[t - 1] = std::thread(work, t);
        } catch (const std::system_error &) {
            // (as many as there are; this thread works too)
        }
        work(0);
        for (std::thread &t : threads)
            if (t.joinable())
                t.join();
        const hipError_t e = hipStreamSynchronize(s);
        return error.load() ? (hipError_t)error.load() : e;
    }
};

struct ffr_renderer {
    std::shared_ptr<HostStage> stage;
    ffr_options opt{};
    FlameSpec spec;
    int mode = MODE_F64_U64;
    int device = 0;
    int cu_count = 256;
    DeviceFlame<double> f64;
    DeviceFlame<float> f32;
    DevTables tab;
    int vs = 2;
    // the wave-per-walker kernel applies: linear variations only (at most
    // kChainSlots per xform), at most four colour dimensions
    bool chain_ok = false;
    bool chain_post_id = false; // ... and every post-affine is the identity
    bool chain_shared = false;  // ... and one pre-affine matrix and weight
    bool chain_diag = false;    // ... and that matrix is diagonal
    size_t chain_lds = 0;       // its LDS bytes
    int chain_per_cu = 0;       // FFR_CHAIN_PER_CU: its walkers-per-CU limit (0: the build's)
    // split walkers apply (no variation draws words, at most four colour
    // dimensions, a rate of contraction that is known or to be expected);
    // the iterations a segment runs before its first, doubled when too many
    // segments of a render entered with another state than the walker's
    bool split_ok = false;
    int split_warm = 0;
    bool last_split = false;
    uint64_t last_split_segments = 0;
    size_t lds_bytes = 0;
    // buffer
    void *dbuf = nullptr;
    uint64_t cells = 0;
    uint32_t cell_words = 1;
    uint32_t word_bytes = 8;
    // statistics
    DevStats *dstats = nullptr;
    unsigned long long *dxf = nullptr;
    unsigned long long *dbv_xfs = nullptr;
    double *dbv_pts = nullptr;
    unsigned long long *dhist = nullptr;
    void *dargs = nullptr;                // the walker kernel's arguments
    unsigned *dhot = nullptr;             // hot-cell hints of the LDS cache
    // streamed buffer I/O: two pinned host chunks, two device chunks
    void *pin[2] = {nullptr, nullptr};
    void *dchunk[2] = {nullptr, nullptr};
    hipEvent_t io_ev[2] = {nullptr, nullptr};
    size_t io_chunk = 0;
    void *dimg = nullptr;                 // image pixels (allocated on first use)
    size_t dimg_bytes = 0;
    std::vector<unsigned char> hargs;     // their host copy, alive until the copy ran
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // the binned walker's probe of the compiled kernel: a pass each
    hipEvent_t ev_ab[4] = {nullptr, nullptr, nullptr, nullptr};
    uint64_t next_walker = 0;
    // cumulative statistics (getters of the reference)
    uint64_t s_iter = 0, s_plot = 0;
    std::vector<uint64_t> xf_dist; // by xform id
    double pmin[3], pmax[3];
    // last render
    uint64_t last_bad = 0, last_walkers = 0, last_batch = 0, last_atomics = 0,
             last_flush_atomics = 0;
    double last_ms = 0;
    std::vector<uint64_t> bv_ids;
    std::vector<double> bv_pts;
    bool pending = false;
    bool timed = false; // ev0/ev1 bracket the pending render (a batch times itself)
    int nxf = 0;
    std::vector<int> order; // sorted position -> xform id
    // launch policy: LDS cell cache (-1 auto, 0 off, 1 on), its LDS budget in
    // KiB, block size (0 auto); FFR_CACHE / FFR_CACHE_KB / FFR_BLOCK override
    int cache_pref = -1;
    int cache_kb = 144;
    int block_pref = 0;
    size_t max_lds = 65536;
    size_t lds_per_cu = 65536;
    int last_cache = 0;
    bool last_chain = false;
    // binned accumulation (-1 chosen per render, 0 off, 1 on where allowed);
    // FFR_BINNED overrides.  Its records, walker states and per-pass
    // arguments are allocated on the first binned render and kept.
    int bin_pref = -1;
    // split walkers: -1 chosen per render, 0 off (FFR_SPLIT)
    int split_pref = -1;
    // miss records: -1 chosen, 0 off, 1 wherever the flame allows them
    // (FFR_MISS); the share of the samples expected to miss the cell cache
    // (measured by each render)
    int miss_pref = -1;
    int task_rounds = 1; // FFR_TASK_ROUNDS: walkers per lane in a task
    RecordLoan records;
    MissTiles miss_tiles;
    double miss_rate = -1;
    // ... without hints (records_args), by log2 of the render's samples
    // (negative: not measured), and of the latest such render; seeded caches
    // miss 0.75 to 0.9 of that, by flame and by run (the 4K colour flame 0.75
    // to 0.88), too wide a range to judge one by the other
    std::vector<double> plain_rates = std::vector<double>(64, -1.0);
    double plain_last = -1;
    int plain_class = -1; // of a render without hints that runs: its log2
    bool last_cached = false; // the last render's misses count (a hashed cache)
    uint64_t last_records = 0; // the last render's misses that became records
    uint32_t last_pauses = 0;  // and the pauses of its workgroups
    BinMemory bin;
    // a colour flame whose renders missed the cell cache often enough
    // (kBinColourRecords, kBinColourAtomics): its later single renders take
    // binned accumulation (binned -1)
    bool bin_colour = false;
    void *wstate = nullptr;
    size_t wstate_bytes = 0;
    void *dargs_bin = nullptr;
    size_t dargs_bin_n = 0;
    bool last_bin = false;
    // the flame compiled into its own kernel (-1 chosen by a probe, 0 off,
    // 1 on); FFR_COMPILED overrides.  rtc_fn: the kernel for the coming
    // launch (nullptr: the table-driven one); compiled_choice: the probe's
    // verdict per launch geometry (cache on/off, lanes per workgroup)
    int compiled_pref = -1;
    void *rtc_fn = nullptr;
    bool last_compiled = false;
    std::unordered_map<int, bool> compiled_choice;
    // cell_cache -1: the probe's verdict per walker count (true: cache kept)
    std::unordered_map<uint64_t, bool> cache_choice;
    // renders launched and samples asked for, over the renderer's life
    uint64_t launches = 0;
    uint64_t samples_asked = 0;
};

// the colour registers of the renderer's walker kernels (the build for three
// is for 2-D flames)
static int walk_nc(const ffr_renderer *r)
{
    const int nc = nc_class(r->spec.color_dims, r->vs);
    return nc == 3 && r->spec.dims != 2 ? 4 : nc;
}

static int pick_variation_set(const uint32_t ts[4])
{
    bool linear_only = true, basic = true;
    for (int t = 0; t < kNumVariations; ++t) {
        if (!(ts[t / 32] >> (t % 32) & 1u))
            continue;
        if (t != 0)
            linear_only = false;
        if (!(t == 0 || t == 1 || t == 2 || t == 20 || t == 21 || t == 22))
            basic = false;
    }
    return linear_only ? 0 : (basic ? 1 : 2);
}

// the settle iterations of a renderer's walkers
template <typename R> static int settle_iterations(const ffr_renderer *r)
{
    return r->opt.settle_iters >= 0 ? (int)r->opt.settle_iters : (sizeof(R) == 4 ? 24 : 53);
}

// Split walkers: how many iterations two trajectories of the flame that draw
// the same words take to become equal bit for bit.  A map that shrinks
// distances by 2^-c on average takes (mantissa bits + a few) / c; the margin
// of 24 covers the spread over trajectories.  For linear flames c comes from
// the maps' largest singular values; other flames are taken to halve a
// distance per iteration (the random flames measured shrink it faster), and
// the device reports where that was wrong.  The colour blend keeps 1 - speed
// of the old colour.  0: the flame does not contract enough.
constexpr int kSplitWarmMax = 512;

template <typename R> static int split_warm_iterations(const DeviceFlame<R> &d, bool linear)
{
    const double bits = (sizeof(R) == 8 ? 53.0 : 24.0) + 24.0;
    const int n = d.dims;
    double map_rate = 0.0, colour_rate = 0.0, before = 0.0;
    for (int x = 0; x < d.nxf; ++x) {
        const double w = (x + 1 < d.nxf ? (double)d.cw[(size_t)x] : 1.0) - before;
        before += w;
        const R *X = d.table.data() + d.xf0 + (size_t)x * (size_t)d.lay.stride;
        if (d.r > 0 && X[d.lay.has_color] != (R)0) {
            const double keep = std::fabs(1.0 - (double)X[d.lay.speed]);
            colour_rate += w * std::min(20.0, -std::log2(std::max(keep, 1e-6)));
        }
        if (!linear)
            continue;
        double wsum = 0.0;
        for (size_t s = 0; s < d.slot_type.size(); ++s)
            if (d.masks[(size_t)x] >> s & 1ull)
                wsum += (double)d.table[(size_t)(d.slot_off[s] + x * d.slot_stride[s])];
        double m[9], mtm[9], v[3] = {1.0, 0.7, 0.4};
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j) {
                m[i * n + j] = 0.0;
                for (int k = 0; k < n; ++k)
                    m[i * n + j] += (double)X[d.lay.postA + i * n + k] * wsum *
                                    (double)X[d.lay.preA + k * n + j];
            }
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j) {
                mtm[i * n + j] = 0.0;
                for (int k = 0; k < n; ++k)
                    mtm[i * n + j] += m[k * n + i] * m[k * n + j];
            }
        // the largest eigenvalue by power iteration
        double norm = 0.0;
        for (int it = 0; it < 32; ++it) {
            double u[3] = {0, 0, 0};
            norm = 0.0;
            for (int i = 0; i < n; ++i) {
                for (int j = 0; j < n; ++j)
                    u[i] += mtm[i * n + j] * v[j];
                norm = std::max(norm, std::fabs(u[i]));
            }
            if (!(norm > 1e-300) || !std::isfinite(norm))
                break;
            for (int i = 0; i < n; ++i)
                v[i] = u[i] / norm;
        }
        if (!std::isfinite(norm))
            return 0;
        map_rate += w * std::min(20.0, -0.5 * std::log2(std::max(norm, 1e-12)));
    }
    double rate = linear ? map_rate : 1.0;
    if (d.r > 0)
        rate = std::min(rate, colour_rate);
    const double k = rate > 0.0 ? std::ceil(bits / rate) : 1e9;
    return k <= (double)kSplitWarmMax ? std::max((int)k, 8) : 0;
}

template <typename R>
static int setup_tables(ffr_renderer *r, const DeviceFlame<R> &d)
{
    if ((int)d.slot_type.size() > kMaxSlots)
        return fail(FFR_E_UNSUPPORTED, "too many variation slots");
    if ((int)d.fin_type.size() > kMaxFinalVars)
        return fail(FFR_E_UNSUPPORTED, "final xform has more than " +
                                           std::to_string(kMaxFinalVars) + " variations");
    if (d.nxf > kMaxXforms)
        return fail(FFR_E_UNSUPPORTED, "more than " + std::to_string(kMaxXforms) + " xforms");
    r->tab.tab_reals = (int)d.table.size();
    r->tab.table_bytes = d.table.size() * sizeof(R);
    HIP_TRY(hipMalloc(&r->tab.table, std::max<size_t>(r->tab.table_bytes, 16)));
    HIP_TRY(hipMemcpy(r->tab.table, d.table.data(), r->tab.table_bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMalloc(&r->tab.masks, sizeof(unsigned long long) * (size_t)d.nxf));
    HIP_TRY(hipMemcpy(r->tab.masks, d.masks.data(), sizeof(unsigned long long) * (size_t)d.nxf,
                      hipMemcpyHostToDevice));
    r->lds_bytes = cache_lds_offset(r->tab.tab_reals, (int)sizeof(R), d.nxf);
    int max_lds = 0;
    HIP_TRY(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock,
                                  r->device));
    if (r->lds_bytes > (size_t)max_lds)
        return fail(FFR_E_UNSUPPORTED, "flame table of " + std::to_string(r->lds_bytes) +
                                           " bytes exceeds the " + std::to_string(max_lds) +
                                           "-byte LDS of a workgroup");
    r->vs = pick_variation_set(d.type_set);
    // the basic set's 2-D kernels add a zero times the mapped point where a
    // list is short, which is nothing while the point is finite
    if (r->vs == 1 && d.dims == 2 && !settles_in_range(d, settle_iterations<R>(r)))
        r->vs = 3;
    r->chain_ok = r->vs == 0 /* linear only, final xform included */ && d.r <= 4 &&
                  d.slot_type.size() <= (size_t)kChainSlots;
    // every xform's post-affine is exactly the identity (entries 1.0 and
    // +0.0, bit for bit): the wave-per-walker kernel then leaves it out (it
    // changes a finite point only in the signs of zeros)
    r->chain_post_id = true;
    for (int x = 0; x < d.nxf && r->chain_post_id; ++x) {
        const R *X = d.table.data() + d.xf0 + (size_t)x * (size_t)d.lay.stride;
        for (int i = 0; i < d.dims * d.dims; ++i) {
            const R v = X[d.lay.postA + i];
            const R want = (i / d.dims == i % d.dims) ? (R)1 : (R)0;
            if (!(v == want && !std::signbit(v)))
                r->chain_post_id = false;
        }
        for (int i = 0; i < d.dims; ++i)
            if (!(X[d.lay.postb + i] == (R)0 && !std::signbit(X[d.lay.postb + i])))
                r->chain_post_id = false;
    }
    // every xform applies the same pre-affine matrix (bit for bit, and in
    // 3-D every one applies it) and one variation of the same weight: the
    // kernel holds them once and broadcasts only the offsets
    r->chain_shared = d.slot_type.size() == 1 && d.nxf > 0;
    for (int x = 0; x < d.nxf && r->chain_shared; ++x) {
        const R *X = d.table.data() + d.xf0 + (size_t)x * (size_t)d.lay.stride;
        const R *X0 = d.table.data() + d.xf0;
        if (std::memcmp(X + d.lay.preA, X0 + d.lay.preA, sizeof(R) * (size_t)(d.dims * d.dims)))
            r->chain_shared = false;
        if (d.dims == 3 && X[d.lay.has_pre] == (R)0)
            r->chain_shared = false;
        if (!(d.masks[(size_t)x] & 1ull))
            r->chain_shared = false;
        const R *w = d.table.data() + d.slot_off[0] + (size_t)x * (size_t)d.slot_stride[0];
        if (std::memcmp(w, d.table.data() + d.slot_off[0], sizeof(R)))
            r->chain_shared = false;
    }
    // the shared matrix is diagonal (off-diagonal entries +0 or -0): the
    // kernel leaves out their products, which are zeros for a finite point
    r->chain_diag = r->chain_shared;
    for (int i = 0; i < d.dims * d.dims && r->chain_diag; ++i)
        if (i / d.dims != i % d.dims && d.table[(size_t)(d.xf0 + d.lay.preA + i)] != (R)0)
            r->chain_diag = false;
    // its LDS: the table, then kChainRows step rows per wave of the flame's
    // build
    const int slots = (int)d.slot_type.size();
    r->chain_lds =
        chain_stage_offset(r->tab.tab_reals, (int)sizeof(R), d.nxf) +
        (size_t)kChainWaves * (size_t)kChainRows * sizeof(R) *
            (size_t)chain_row_reals((int)sizeof(R), d.dims, d.r > 0 ? 4 : 0, chain_build_ns(slots),
                                    r->chain_post_id,
                                    chain_build_sh(r->chain_shared, r->chain_post_id, slots));
    if (r->chain_lds > (size_t)max_lds)
        r->chain_ok = false;
    r->split_ok = d.r <= 4 && d.nxf > 0;
    for (int t : d.slot_type)
        r->split_ok = r->split_ok && variation_draws(t, d.dims) == 0;
    for (int t : d.fin_type)
        r->split_ok = r->split_ok && variation_draws(t, d.dims) == 0;
    if (r->split_ok)
        r->split_warm = split_warm_iterations(d, r->vs == 0);
    r->split_ok = r->split_ok && r->split_warm > 0;
    r->nxf = d.nxf;
    r->order = d.order;
    return FFR_OK;
}

extern "C" {

void ffr_default_options(ffr_options *opt)
{
    if (!opt)
        return;
    std::memset(opt, 0, sizeof *opt);
    opt->precision = FFR_FP64;
    opt->word = FFR_WORD64;
    opt->settle_iters = -1;
    opt->bad_value_limit = 256;
    opt->bad_value_cap = 4096;
    opt->cell_cache = -1;
    opt->binned = -1;
    opt->compiled = -1;
}

const char *ffr_last_error(void) { return g_err.c_str(); }

int ffr_create(const char *flame_json, size_t len, const ffr_options *opt_in,
               ffr_renderer **out)
{
    if (!flame_json || !out)
        return fail(FFR_E_ARG, "ffr_create: null argument");
    *out = nullptr;
    ffr_options opt;
    if (opt_in)
        opt = *opt_in;
    else
        ffr_default_options(&opt);
    if (opt.precision > FFR_FP32 || opt.word > FFR_WORD32)
        return fail(FFR_E_ARG, "ffr_create: unknown precision or word option");
    if (opt.precision == FFR_FP64 && opt.word == FFR_WORD32)
        return fail(FFR_E_UNSUPPORTED,
                    "FP64 trajectories need 64-bit buffer words (sizeof(num_t) == sizeof(hist_t))");
    if (opt.bad_value_cap == 0)
        opt.bad_value_cap = 4096;
    std::unique_ptr<ffr_renderer> r(new ffr_renderer());
    r->opt = opt;
    r->device = opt.device;
    r->stage = HostStage::of_device(opt.device);
    r->records.open(opt.device);
    r->mode = opt.precision == FFR_FP64 ? MODE_F64_U64
                                        : (opt.word == FFR_WORD32 ? MODE_F32_U32 : MODE_F32_U64);
    const bool fp32 = opt.precision == FFR_FP32;
    try {
        Json doc = Json::parse(std::string(flame_json, len));
        r->spec = parse_flame(doc, fp32);
        if (fp32)
            r->f32 = compile_flame<float>(r->spec);
        else
            r->f64 = compile_flame<double>(r->spec);
    } catch (const std::exception &e) {
        return fail(FFR_E_FLAME, e.what());
    }
    {
        const XformLayout &lay = fp32 ? r->f32.lay : r->f64.lay;
        if (!layout_matches_kernels(lay, r->spec.dims))
            return fail(FFR_E_UNSUPPORTED, "ffr_create: xform record layout differs from the kernels'");
    }
    HIP_TRY(hipSetDevice(r->device));
    HIP_TRY(hipDeviceGetAttribute(&r->cu_count, hipDeviceAttributeMultiprocessorCount,
                                  r->device));
    {
        int v = 0;
        HIP_TRY(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, r->device));
        r->max_lds = (size_t)v;
        v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor,
                                  r->device) == hipSuccess && v > 0)
            r->lds_per_cu = (size_t)v;
        else
            r->lds_per_cu = r->max_lds;
        r->cache_pref = opt.cell_cache < 0 ? -1 : (opt.cell_cache ? 1 : 0);
        if (opt.cache_kib > 0)
            r->cache_kb = opt.cache_kib;
        if (opt.block > 0)
            r->block_pref = opt.block;
        if (const char *e = std::getenv("FFR_CACHE"))
            r->cache_pref = std::atoi(e);
        if (const char *e = std::getenv("FFR_CACHE_KB"))
            r->cache_kb = std::max(1, std::atoi(e));
        if (const char *e = std::getenv("FFR_BLOCK"))
            r->block_pref = std::atoi(e);
        r->bin_pref = opt.binned < 0 ? -1 : (opt.binned ? 1 : 0);
        if (const char *e = std::getenv("FFR_BINNED"))
            r->bin_pref = std::atoi(e);
        if (const char *e = std::getenv("FFR_SPLIT"))
            r->split_pref = std::atoi(e) ? -1 : 0;
        if (const char *e = std::getenv("FFR_MISS"))
            r->miss_pref = std::atoi(e) < 0 ? -1 : (std::atoi(e) ? 1 : 0);
        r->compiled_pref = opt.compiled < 0 ? -1 : (opt.compiled ? 1 : 0);
        if (const char *e = std::getenv("FFR_TASK_ROUNDS"))
            r->task_rounds = std::max(1, std::atoi(e));
        if (const char *e = std::getenv("FFR_CHAIN_PER_CU"))
            r->chain_per_cu = std::atoi(e);
        if (const char *e = std::getenv("FFR_COMPILED"))
            r->compiled_pref = std::atoi(e) < 0 ? -1 : (std::atoi(e) ? 1 : 0);
    }
    int rc = fp32 ? setup_tables(r.get(), r->f32) : setup_tables(r.get(), r->f64);
    if (rc != FFR_OK) {
        ffr_destroy(r.release());
        return rc;
    }
    r->cells = r->spec.cells();
    r->cell_words = 1u + (uint32_t)r->spec.color_dims;
    r->word_bytes = r->mode == MODE_F32_U32 ? 4u : 8u;
    const size_t bytes = (size_t)r->cells * r->cell_words * r->word_bytes;
    hipError_t e = device_malloc(&r->dbuf, bytes);
    if (e != hipSuccess) {
        ffr_destroy(r.release());
        return fail(FFR_E_DEVICE, "hipMalloc of the " + std::to_string(bytes) +
                                      "-byte buffer: " + hipGetErrorString(e));
    }
    ffr_renderer *rp = r.release();
#define HIP_TRY_D(call)                                                                \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess) {                                                        \
            ffr_destroy(rp);                                                           \
            return fail(FFR_E_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
        }                                                                              \
    } while (0)
    HIP_TRY_D(hipStreamCreateWithFlags(&rp->own_stream, hipStreamNonBlocking));
    rp->stream = rp->own_stream;
    HIP_TRY_D(hipEventCreate(&rp->ev0));
    HIP_TRY_D(hipEventCreate(&rp->ev1));
    HIP_TRY_D(hipMalloc(&rp->dstats, (1 + kSplitSlots) * sizeof(DevStats)));
    HIP_TRY_D(hipMalloc(&rp->dxf, 2 * sizeof(unsigned long long) * (size_t)std::max(rp->nxf, 1)));
    HIP_TRY_D(hipMalloc(&rp->dbv_xfs, sizeof(unsigned long long) * rp->opt.bad_value_cap));
    HIP_TRY_D(hipMalloc(&rp->dbv_pts, sizeof(double) * 3 * rp->opt.bad_value_cap));
    HIP_TRY_D(hipMalloc(&rp->dhist, sizeof(unsigned long long) * (kHistWords + kToneLut)));
    // (two: a split launch's and those of the launch behind it)
    HIP_TRY_D(hipMalloc(&rp->dargs,
                        2 * std::max(sizeof(WalkArgs<double>), sizeof(WalkArgs<float>))));
    // hints start empty: a tag no geometry has
    HIP_TRY_D(hipMalloc(&rp->dhot, sizeof(unsigned) * (1 + (size_t)kHotSlots)));
    HIP_TRY_D(hipMemsetAsync(rp->dhot, 0xFF, sizeof(unsigned) * (1 + (size_t)kHotSlots),
                             rp->stream));
    HIP_TRY_D((hipError_t)launch_fill_zero(rp->dbuf, bytes, rp->stream));
    HIP_TRY_D(hipStreamSynchronize(rp->stream));
#undef HIP_TRY_D
    rp->xf_dist.assign(rp->spec.xforms.size(), 0);
    for (int i = 0; i < 3; ++i) {
        rp->pmin[i] = INFINITY;
        rp->pmax[i] = -INFINITY;
    }
    *out = rp;
    return FFR_OK;
}

void ffr_destroy(ffr_renderer *r)
{
    if (!r)
        return;
    // teardown: errors here have nowhere to go
    (void)hipSetDevice(r->device);
    if (r->own_stream)
        (void)hipStreamSynchronize(r->own_stream);
    if (r->stream && r->stream != r->own_stream)
        (void)hipStreamSynchronize(r->stream);
    (void)hipFree(r->tab.table);
    (void)hipFree(r->tab.masks);
    (void)hipFree(r->dbuf);
    (void)hipFree(r->dstats);
    (void)hipFree(r->dxf);
    (void)hipFree(r->dbv_xfs);
    (void)hipFree(r->dbv_pts);
    (void)hipFree(r->dhist);
    (void)hipFree(r->dargs);
    (void)hipFree(r->dimg);
    (void)hipFree(r->dhot);
    r->bin.free_all();
    (void)hipFree(r->wstate);
    (void)hipFree(r->dargs_bin);
    r->records.give_back();
    r->miss_tiles.free_all();
    for (int k = 0; k < 2; ++k) {
        if (r->pin[k])
            (void)hipHostFree(r->pin[k]);
        (void)hipFree(r->dchunk[k]);
        if (r->io_ev[k])
            (void)hipEventDestroy(r->io_ev[k]);
    }
    if (r->ev0)
        (void)hipEventDestroy(r->ev0);
    if (r->ev1)
        (void)hipEventDestroy(r->ev1);
    for (hipEvent_t ev : r->ev_ab)
        if (ev)
            (void)hipEventDestroy(ev);
    if (r->own_stream)
        (void)hipStreamDestroy(r->own_stream);
    delete r;
}

uint64_t ffr_auto_batch(const ffr_renderer *r, uint64_t samples)
{
    (void)r;
    // enough walkers to fill the device (about 2^19 lanes), each long
    // enough that its settle iterations stay a small share of its work
    const uint64_t target_walkers = 1ull << 19;
    uint64_t b = (samples + target_walkers - 1) / target_walkers;
    if (b < 1024)
        b = 1024;
    return b;
}

} // extern "C"

template <typename R>
static void fill_args(ffr_renderer *r, const DeviceFlame<R> &d, WalkArgs<R> &a)
{
    std::memset(&a, 0, sizeof a);
    a.table = (const R *)r->tab.table;
    a.masks = r->tab.masks;
    a.buf = r->dbuf;
    a.stats = r->dstats;
    a.xf_count = r->dxf;
    a.bv_xfs = r->dbv_xfs;
    a.bv_pts = r->dbv_pts;
    for (int i = 0; i < 3; ++i) {
        a.lo[i] = d.lo[i];
        a.hi[i] = d.hi[i];
        a.mult_d[i] = d.mult_d[i];
        a.mult_i[i] = d.mult_i[i];
    }
    a.cells = d.cells;
    a.seed = r->opt.seed;
    a.bv_limit = r->opt.bad_value_limit;
    a.bv_cap = r->opt.bad_value_cap;
    a.nxf = d.nxf;
    a.n_slots = (int)d.slot_type.size();
    a.has_final = d.has_final;
    a.fin_nv = (int)d.fin_type.size();
    a.settle = settle_iterations<R>(r);
    a.r = d.r;
    a.tab_reals = (int)d.table.size();
    a.xf0 = d.xf0;
    a.fin0 = d.fin0;
    a.l_preA = d.lay.preA;
    a.l_preb = d.lay.preb;
    a.l_postA = d.lay.postA;
    a.l_postb = d.lay.postb;
    a.l_speed = d.lay.speed;
    a.l_color = d.lay.color;
    a.l_has_color = d.lay.has_color;
    a.l_has_pre = d.lay.has_pre;
    a.l_has_post = d.lay.has_post;
    a.l_stride = d.lay.stride;
    for (size_t s = 0; s < d.slot_type.size(); ++s) {
        a.slot_type[s] = d.slot_type[s];
        a.slot_off[s] = d.slot_off[s];
        a.slot_stride[s] = d.slot_stride[s];
    }
    a.bt0 = d.bt0;
    a.bt_stride = d.bt_stride;
    a.bt_nvmax = d.bt_nvmax;
    a.bt_union = d.bt_union;
    for (size_t j = 0; j < d.fin_type.size(); ++j) {
        a.fin_type[j] = d.fin_type[j];
        a.fin_off[j] = d.fin_off[j];
    }
}

// launch shape: what the launch may use; results do not depend on it
struct LaunchShape {
    int cache = -1;     // LDS cell cache: -1 chosen, 0 off, 1 on
    int cache_kb = 144; // LDS budget of the cache per workgroup, KiB
    int block = 0;      // lanes per workgroup, 0 chosen
    int task_rounds = 1; // walkers per lane in one workgroup task
    int bin = -1;       // binned accumulation (single renders): -1 chosen, 0 off, 1 on
    int split = 0;      // split walkers (single renders): -1 chosen, 0 off
};

static LaunchShape renderer_shape(const ffr_renderer *r)
{
    LaunchShape sh;
    sh.bin = r->bin_pref;
    sh.split = r->split_pref;
    sh.task_rounds = r->task_rounds;
    sh.cache = r->cache_pref;
    sh.cache_kb = r->cache_kb;
    sh.block = r->block_pref;
    return sh;
}

// launch geometry of one render pass (see plan_launch)
struct LaunchPlan {
    bool chain = false; // one walker per wave (chain_kernel)
    bool bin = false;   // binned accumulation (walk_bin_kernel + bin_kernels)
    int split_log2 = 0; // split walkers: log2 of the segments per walker (0: not split)
    uint64_t split_len = 0;     // iterations per segment
    bool cache = false;
    int block = 256;
    int grid = 1;
    size_t lds = 0;
    int slots = 0, log2s = 0, ways = 1, direct = 0;
    uint64_t task_walkers = 256;
};

static size_t table_lds(const ffr_renderer *r)
{
    const int rb = r->mode == MODE_F64_U64 ? 8 : 4;
    return cache_lds_offset(r->tab.tab_reals, rb, r->nxf);
}

// Split walkers (split_kernel.inc): renders of few walkers, whose unsplit
// launches are bound by the chain of one walker's iterations, and without
// the LDS cell cache (off below 64 walkers per CU) by atomics on hot cells.
// A walker is split into a power of two of segments, as many as fill the
// device (4 waves per SIMD; measured at 2^26 samples of 1024 walkers: 65536
// lanes 3.9 ms, 131072 2.9, 262144 2.6, 524288 2.6) while a segment keeps 16
// iterations (2^20 samples: 8 iterations 0.29-0.33 ms, 16 0.26-0.29, 64
// 0.33, 256 0.72).  Kernel time of one render, unsplit then split:
//   256^2 colour flame, 1024 walkers x 1024, FP32            8.8 -> 0.22 ms
//   1024^2 colour flame, 1024 walkers x 65536, FP32        145   -> 2.6 ms
//   Sierpinski 1024^2, 1024 x 65536, FP64 (wave per walker)  4.8 -> 1.1 ms
//   3-D linear flame, 1892 walkers x 1024, FP32              5.4 -> 0.26 ms
// The smallest of the renders tried, 1400 walkers x 1024 of a triangle, goes
// from 0.30 to 0.20 ms.
static void split_plan(const ffr_renderer *r, uint64_t walkers, uint64_t batch,
                       const LaunchShape &sh, bool chain, LaunchPlan &p)
{
    const int ncol = r->spec.color_dims;
    if (sh.split >= 0 || !r->split_ok || sh.cache >= 0 || sh.block > 0 || sh.bin >= 0)
        return;
    if (!chain && (r->compiled_pref > 0 || walkers >= (uint64_t)r->cu_count * 64u))
        return;
    if (r->cells >= (ncol > 0 ? (1ull << 25) : (1ull << 28)))
        return;
    // (float colour sums of 4-byte words keep the per-sample float adds of
    // the unsplit kernels: added in double per tile they come out closer to
    // the true sums, but elsewhere than the float build's own)
    if (ncol > 0 && r->word_bytes == 4)
        return;
    const uint64_t lanes = (uint64_t)r->cu_count * 1024u;
    int log2s = 0;
    while (log2s < kSplitMaxLog2 && (walkers << (log2s + 1)) <= lanes &&
           (batch >> (log2s + 1)) >= 16)
        ++log2s;
    if (log2s == 0)
        return;
    // (an even length: the segments' words then start alike in a block)
    const uint64_t len = (((batch + (1ull << log2s) - 1) >> log2s) + 1) & ~1ull;
    const uint64_t per_group = (uint64_t)kSplitBlock >> log2s; // walkers per workgroup
    const uint64_t groups = (walkers + per_group - 1) / per_group;
    if (len > kBinPassRecords / kSplitBlock || groups * kSplitBlock > kBinPassRecords / len)
        return;
    p.split_log2 = log2s;
    p.split_len = len;
}

// Accumulation through the LDS cell cache needs cell indices below 2^32,
// at most 4 colour words, and per-task counts that fit 32 bits (a task of
// task_walkers walkers adds at most task_walkers * batch to one cell).  The
// cache takes the LDS left after the flame table, up to the budget; a
// buffer that fits entirely is indexed directly.  `base_lds` is the LDS the
// launch must hold besides the cache (the largest flame table of a batch).
static LaunchPlan plan_launch(const ffr_renderer *r, uint64_t walkers, uint64_t batch,
                              const LaunchShape &sh, size_t base_lds = 0)
{
    LaunchPlan p;
    const size_t base = std::max(table_lds(r), base_lds);
    const int per_cu = r->chain_per_cu > 0
                           ? r->chain_per_cu
                           : chain_walkers_per_cu(r->chain_post_id, r->spec.color_dims);
    const bool chain = sh.cache < 0 && sh.block <= 0 && base_lds == 0 && r->chain_ok &&
                       walkers <= (uint64_t)r->cu_count * (uint64_t)per_cu;
    // binned accumulation: single renders whose walkers all fit one pass's
    // records, of count-only buffers under 2^28 cells or colour buffers (up
    // to four colour dimensions) under 2^25; chosen for count-only buffers
    // from 2^22 cells on when the lane-per-walker kernel runs (the samples
    // spread beyond what an LDS cache holds), for colour flames whose
    // earlier renders spent many global atomics per sample (bin_colour),
    // or when asked for
    const uint64_t tw_bin = (uint64_t)kBinWalkBlock;
    const int ncol = r->spec.color_dims;
    if (base_lds == 0)
        split_plan(r, walkers, batch, sh, chain, p);
    if (p.split_log2) {
        p.chain = chain; // (the launch behind it)
        p.block = kSplitBlock;
        p.task_walkers = (uint64_t)kSplitBlock >> p.split_log2;
        p.grid = (int)((walkers + p.task_walkers - 1) / p.task_walkers);
        const int rb = r->mode == MODE_F64_U64 ? 8 : 4;
        p.lds = split_lds(base, rb, r->spec.dims, ncol > 0 ? 4 : 0);
        if (p.lds <= r->max_lds)
            return p;
        p = LaunchPlan();
    }
    const bool bin_ok = base_lds == 0 && ncol <= 4 &&
                        r->cells < (ncol > 0 ? (1ull << 25) : (1ull << 28)) &&
                        (walkers + tw_bin - 1) / tw_bin * tw_bin <= kBinPassRecords;
    const bool bin_auto = sh.bin < 0 && !chain && sh.cache < 0 && sh.block <= 0 &&
                          (ncol == 0 ? r->cells >= (1ull << 22) : r->bin_colour);
    if (bin_ok && (sh.bin == 1 || bin_auto)) {
        p.bin = true;
        p.block = kBinWalkBlock;
        p.task_walkers = tw_bin;
        p.grid = (int)std::min<uint64_t>((walkers + tw_bin - 1) / tw_bin, 1u << 30);
        p.lds = base;
        (void)batch;
        return p;
    }
    // few walkers of a linear flame: one walker per wave, its chain split
    // into parallel draws and plots around a short serial part (unless the
    // cache or the workgroup size is forced)
    if (chain) {
        p.chain = true;
        p.block = 64 * kChainWaves;
        p.task_walkers = (uint64_t)kChainWaves;
        p.grid = (int)((walkers + kChainWaves - 1) / kChainWaves);
        p.lds = r->chain_lds; // the table, then each wave's 64 step rows
        return p;
    }
    const int colour_bytes = r->word_bytes;
    const size_t slot_bytes = cache_slot_bytes(r->spec.color_dims, colour_bytes);
    bool want = sh.cache != 0 && r->cells < 0xFFFFFFFFull && r->spec.color_dims <= 4;
    // with fewer walkers than one wave per CU the render is bound by the
    // latency of one walker's chain, which the cache lengthens (unless
    // forced on); from there on the cache keeps hot cells off the device's
    // atomics (measured: 64000 walkers on a 256^2 flame, 0.12 G samples/s
    // without it, 16 with it)
    if (sh.cache < 0 && walkers < (uint64_t)r->cu_count * 64u)
        want = false;
    const int bmax = cache_block_max(r->mode == MODE_F64_U64, r->vs);
    p.block = (sh.block > 0 && sh.block <= bmax) ? sh.block : bmax;
    const uint64_t rounds = (uint64_t)std::max(1, sh.task_rounds);
    if (want && (uint64_t)p.block * batch >= (1ull << 31))
        want = false;
    if (want) {
        // (256 bytes stay free for the batched kernel's static LDS)
        size_t budget = std::min<size_t>(r->max_lds - 256, (size_t)sh.cache_kb << 10);
        size_t avail = budget > base ? budget - base : 0;
        int log2s = 0;
        while (((size_t)2 << log2s) * slot_bytes <= avail && log2s < 30)
            ++log2s;
        if (((size_t)1 << log2s) * slot_bytes > avail)
            want = false;
        else {
            p.log2s = log2s;
            p.slots = 1 << log2s;
            p.ways = 4;
            if ((uint64_t)p.slots >= r->cells) {
                while (p.log2s > 0 && ((uint64_t)1 << (p.log2s - 1)) >= r->cells)
                    --p.log2s;
                p.slots = 1 << p.log2s;
                p.direct = 1;
                p.ways = 1;
            }
        }
    }
    p.cache = want;
    if (p.cache) {
        p.lds = base + (size_t)p.slots * slot_bytes;
        uint64_t rr = std::min<uint64_t>(rounds, ((1ull << 31) - 1) / ((uint64_t)p.block * batch));
        p.task_walkers = (uint64_t)p.block * std::max<uint64_t>(rr, 1);
        int per_cu = std::max<int>(1, (int)(r->lds_per_cu / std::max<size_t>(p.lds, 1)));
        uint64_t tasks = (walkers + p.task_walkers - 1) / p.task_walkers;
        p.grid = (int)std::max<uint64_t>(
            1, std::min<uint64_t>(tasks, (uint64_t)r->cu_count * (uint64_t)per_cu));
    } else {
        p.block = walkers >= (uint64_t)r->cu_count * 256 ? 256 : 64;
        if (sh.block > 0 && sh.block <= 256)
            p.block = sh.block;
        p.task_walkers = (uint64_t)p.block * rounds;
        uint64_t tasks = (walkers + p.task_walkers - 1) / p.task_walkers;
        p.grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(tasks, 1u << 30));
        p.lds = base;
    }
    return p;
}

template <typename R>
static void walk_args(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan &p,
                      uint64_t walker0, uint64_t n_walkers, uint64_t batch, uint64_t last,
                      WalkArgs<R> &a, bool hints = false)
{
    fill_args(r, d, a);
    a.walker_base = walker0;
    a.n_walkers = n_walkers;
    a.batch = batch;
    a.last_samples = last;
    a.task_walkers = p.task_walkers;
    a.cache_slots = p.slots;
    a.cache_log2 = p.log2s;
    a.cache_ways = p.ways;
    a.cache_direct = p.direct;
    // hot-cell hints for hashed caches (a task keeps a slot as a hint when
    // it counted at least an eighth of its samples per slot there, and at
    // least hot_thresh); the tag names the cache geometry of the hints.
    // Only for flames that few workgroups render at once: workgroups seeded
    // alike miss the same cells, and their global atomics then queue on the
    // same addresses (the headline flame on all 256 CUs ran 3x slower).
    a.hot = nullptr;
    a.hot_tag = 0;
    a.hot_thresh = 2;
    if (hints && p.cache && !p.direct && p.slots <= kHotSlots && r->dhot) {
        a.hot = r->dhot;
        a.hot_tag = 0x40000000u | ((unsigned)p.log2s << 8) | (unsigned)p.ways;
    }
}

static int launch_walk_any(int mode, int dims, const WalkLaunch &L)
{
    if (L.split)
        switch (mode) {
        case MODE_F64_U64:
            return dims == 1 ? launch_split_f64u64_d1(L) : dims == 2 ? launch_split_f64u64_d2(L)
                                                                      : launch_split_f64u64_d3(L);
        case MODE_F32_U32:
            return dims == 1 ? launch_split_f32u32_d1(L) : dims == 2 ? launch_split_f32u32_d2(L)
                                                                      : launch_split_f32u32_d3(L);
        default:
            return dims == 1 ? launch_split_f32u64_d1(L) : dims == 2 ? launch_split_f32u64_d2(L)
                                                                      : launch_split_f32u64_d3(L);
        }
    switch (mode) {
    case MODE_F64_U64:
        return dims == 1 ? launch_walk_f64u64_d1(L) : dims == 2 ? launch_walk_f64u64_d2(L)
                                                                 : launch_walk_f64u64_d3(L);
    case MODE_F32_U32:
        return dims == 1 ? launch_walk_f32u32_d1(L) : dims == 2 ? launch_walk_f32u32_d2(L)
                                                                 : launch_walk_f32u32_d3(L);
    default:
        return dims == 1 ? launch_walk_f32u64_d1(L) : dims == 2 ? launch_walk_f32u64_d2(L)
                                                                 : launch_walk_f32u64_d3(L);
    }
}

static int launch_walk_any(int mode, int dims, const WalkLaunch &L);

// the table-driven walker kernel for a plan, its arguments at `dargs`
static int launch_table_kernel(ffr_renderer *r, const LaunchPlan &p, int nslots,
                               const void *dargs)
{
    WalkLaunch L;
    L.nc = r->spec.color_dims;
    L.vs = r->vs;
    L.chain = p.chain;
    L.chain_slots = nslots;
    L.chain_post_id = r->chain_post_id;
    L.chain_shared = r->chain_shared;
    L.chain_diag = r->chain_diag;
    L.cache = p.cache;
    L.grid = p.grid;
    L.block = p.block;
    L.lds = p.lds;
    L.stream = r->stream;
    L.args = dargs;
    return launch_walk_any(r->mode, r->spec.dims, L);
}

// the flame's compiled kernel, its arguments (the WalkDyn part) at `dargs`
static int launch_compiled_kernel(ffr_renderer *r, const LaunchPlan &p, void *fn,
                                  const void *dargs)
{
    void *params[] = {&dargs};
    return (int)hipModuleLaunchKernel((hipFunction_t)fn, (unsigned)p.grid, 1, 1,
                                      (unsigned)p.block, 1, 1, (unsigned)p.lds, r->stream,
                                      params, nullptr);
}

// With compiled -1 a renderer in steady use (its second render or later,
// once its renders have asked for this many samples in all) compiles the
// flame's kernel and probes whether it beats the table-driven one: the
// compile (about half a second) pays off only over repeated renders.
constexpr uint64_t kCompiledProbeSamples = 1ull << 33;

// the lanes of a cached plan that the device holds at a time
static uint64_t cached_lanes(const ffr_renderer *r, const LaunchPlan &p)
{
    const uint64_t groups = std::max<uint64_t>(1, r->lds_per_cu / std::max<size_t>(p.lds, 1));
    return (uint64_t)r->cu_count * groups * (uint64_t)p.block;
}

// Miss records apply to a cached launch of a flame whose cells (and colour
// sums) the binning kernels hold: not colour flames with 4-byte words, whose
// float sums keep the per-sample float adds
static bool miss_ok(const ffr_renderer *r)
{
    const int ncol = r->spec.color_dims;
    return r->miss_pref != 0 && ncol <= 4 && !(ncol > 0 && r->word_bytes == 4) &&
           r->cells < (ncol > 0 ? (1ull << 25) : (1ull << 28));
}

// The share of a render's samples that its launch would miss without hints,
// as far as earlier renders tell
static int rate_class(uint64_t samples)
{
    return 63 - __builtin_clzll(samples | 1);
}

static double plain_rate(const ffr_renderer *r, uint64_t samples)
{
    const double known = r->plain_rates[rate_class(samples)];
    return known >= 0 ? known : r->plain_last;
}

// ... and are taken by a launch of enough walkers and samples that miss
// enough (not where the cache is forced, or indexed directly, so that
// nothing misses; their memory may be allocated, so not while the stream is
// captured)
static bool records_wanted(const ffr_renderer *r, const LaunchPlan &p, uint64_t walkers,
                           uint64_t batch, int real_bytes)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    return p.cache && !p.direct && r->cache_pref < 0 && miss_ok(r) &&
           (r->miss_pref > 0 ||
            (miss_worth(plain_rate(r, walkers * batch), (int)r->cell_words, real_bytes, false,
                        walkers, cached_lanes(r, p)) &&
             walkers * batch >= kMissMinSamples)) &&
           hipStreamIsCapturing(r->stream, &cap) == hipSuccess &&
           cap == hipStreamCaptureStatusNone;
}

// The memory for the records of a launch into `buf`, and its rounds: none
// without the memory (the misses then stay atomics).
static int reserve_records(ffr_renderer *r, const LaunchPlan &p, uint64_t walkers, uint64_t batch,
                           int real_bytes, void *buf, MissTiles &tiles, MissRounds &m)
{
    m = MissRounds();
    if (const int rc = prepare_miss_once())
        return rc;
    const int words = record_words(walk_nc(r), real_bytes);
    MissMemory &mem = r->records.get().miss;
    MissRounds want =
        miss_rounds(mem, walkers * batch,
                    (walkers + p.task_walkers - 1) / p.task_walkers, p.grid, p.block, words,
                    r->miss_rate);
    if (!want.rounds)
        return 0;
    hipError_t e = mem.ensure(p.grid, p.block, want.chunks, words, real_bytes);
    if (e == hipSuccess) {
        MissFlame f{};
        f.buf = buf;
        f.cells = r->cells;
        f.r = r->spec.color_dims;
        e = tiles.set({f}, f.r > 0 ? kBinTileBitsColour : kBinTileBits, r->stream);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        mem.free_all();
        return 0;
    }
    m = want;
    return 0;
}

static MissScratch records_scratch(const ffr_renderer *r, const LaunchPlan &p,
                                   const MissTiles &tiles, const MissRounds &m, int real_bytes)
{
    return miss_scratch(r->records.mem->miss, tiles, m.chunks, p.grid,
                        record_words(walk_nc(r), real_bytes), real_bytes, r->cu_count);
}

// the arguments of a lane-per-walker render of `samples`: its walker
// launches', and those of the last one, which has no record memory
template <typename R>
static void records_args(const ffr_renderer *r, const LaunchPlan &p, const MissTiles &tiles,
                         const MissRounds &m, uint64_t samples, WalkArgs<R> (&a)[2])
{
    if (m.rounds) {
        a[0].miss = miss_args(records_scratch(r, p, tiles, m, (int)sizeof(R)), m.limit);
        // hints: with records, workgroups seeded alike have no atomics to
        // queue on (the headline flame misses 3.0 instead of 3.5 %), once a
        // render of this size went without (55.9 instead of 55.2 ms) and
        // left the rate that its records are judged by
        if (r->dhot && p.slots <= kHotSlots && r->plain_rates[rate_class(samples)] >= 0) {
            a[0].hot = r->dhot;
            a[0].hot_tag = 0x40000000u | ((unsigned)p.log2s << 8) | (unsigned)p.ways;
        }
    }
    a[1] = a[0];
    a[1].miss.chunks = 0;
}

// the launches of such a render, by the flame's compiled kernel fn or the
// table-driven one (nullptr); the arguments are at r->dargs
template <typename R>
static int launch_rounds(ffr_renderer *r, const LaunchPlan &p, void *fn, int nslots,
                         const MissTiles &tiles, const MissRounds &m)
{
    // (a compiled flame's kernel reads only the launch part, WalkDyn, at the
    // start of WalkArgs; its flame fields are constants)
    auto walk = [&](int k) {
        const void *args = (const unsigned char *)r->dargs + (size_t)k * sizeof(WalkArgs<R>);
        return fn ? launch_compiled_kernel(r, p, fn, args)
                  : launch_table_kernel(r, p, nslots, args);
    };
    if (!m.rounds)
        return walk(0);
    const MissScratch x = records_scratch(r, p, tiles, m, (int)sizeof(R));
    int rc = launch_miss_init(x, p.task_walkers, r->stream);
    for (int k = 0; k < m.rounds && !rc; ++k) {
        rc = walk(0);
        if (!rc)
            rc = launch_miss_round(x, (int)r->word_bytes, r->stream);
    }
    if (!rc && m.last)
        rc = walk(1);
    return rc;
}

// Time kernels for the coming render: n launch plans, each with the flame's
// compiled kernel fns[k] or the table-driven one (nullptr), on the render's
// walkers with at most 1024 samples each, into a scratch buffer: the
// renderer's buffer and stream positions are untouched, and the statistics
// the runs leave are reset before the render.  Misses become records where
// the render's would, and their binning is timed with the walkers.  ms[k]: the better of two
// runs (one, when after the first every other kernel took more than
// stop_ratio times kernel 0's time; 0: always two).
template <typename R>
static int time_kernels(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan *plans,
                        void *const *fns, int n, uint64_t walker0, uint64_t walkers,
                        uint64_t batch, float *ms, float stop_ratio = 0.f)
{
    const uint64_t pb = std::min<uint64_t>(batch, 1024);
    void *scratch = nullptr;
    HIP_TRY(device_malloc(&scratch, ffr_buffer_bytes(r)));
    std::vector<std::vector<unsigned char>> h((size_t)n);
    std::vector<MissRounds> rounds((size_t)n);
    MissTiles tiles;
    for (int k = 0; k < n; ++k) {
        ms[k] = 1e30f;
        int rc = 0;
        if (records_wanted(r, plans[k], walkers, batch, (int)sizeof(R)))
            rc = reserve_records(r, plans[k], walkers, pb, (int)sizeof(R), scratch, tiles,
                                 rounds[(size_t)k]);
        if (rc) {
            tiles.free_all();
            (void)hipFree(scratch);
            return fail(FFR_E_DEVICE, std::string("kernel probe: ") +
                                          hipGetErrorString((hipError_t)rc));
        }
    }
    // (the record memory stands now)
    for (int k = 0; k < n; ++k) {
        WalkArgs<R> a[2];
        walk_args(r, d, plans[k], walker0, walkers, pb, pb, a[0]);
        a[0].buf = scratch;
        a[0].bv_limit = ~0ull; // the runs never stop at the bad-value limit
        records_args(r, plans[k], tiles, rounds[(size_t)k], walkers * batch, a);
        h[(size_t)k].resize(sizeof a);
        std::memcpy(h[(size_t)k].data(), a, sizeof a);
    }
    hipError_t e = hipSuccess;
    for (int round = 0; round < 2 && e == hipSuccess; ++round) {
        if (round == 1 && stop_ratio > 0.f) {
            bool all_slower = true;
            for (int k = 1; k < n; ++k)
                all_slower = all_slower && ms[k] > stop_ratio * ms[0];
            if (all_slower)
                break;
        }
        for (int k = 0; k < n && e == hipSuccess; ++k) {
            e = hipMemcpyAsync(r->dargs, h[(size_t)k].data(), h[(size_t)k].size(),
                               hipMemcpyHostToDevice, r->stream);
            if (e == hipSuccess)
                e = launch_reset_stats(r->dstats, r->dxf, r->nxf, r->stream)
                        ? hipErrorLaunchFailure
                        : hipSuccess;
            if (e == hipSuccess)
                e = hipEventRecord(r->ev0, r->stream);
            if (e == hipSuccess)
                e = (hipError_t)launch_rounds<R>(r, plans[k], fns[k], (int)d.slot_type.size(),
                                                 tiles, rounds[(size_t)k]);
            if (e == hipSuccess)
                e = hipEventRecord(r->ev1, r->stream);
            if (e == hipSuccess)
                e = hipEventSynchronize(r->ev1);
            float t = 0;
            if (e == hipSuccess)
                e = hipEventElapsedTime(&t, r->ev0, r->ev1);
            if (e == hipSuccess)
                ms[k] = std::min(ms[k], t);
        }
    }
    const hipError_t ef = hipFree(scratch);
    tiles.free_all();
    if (e == hipSuccess)
        e = ef;
    if (e != hipSuccess)
        return fail(FFR_E_DEVICE, std::string("kernel probe: ") + hipGetErrorString(e));
    return FFR_OK;
}

// With the cell cache left to the renderer (cell_cache -1), a renderer in
// steady use (its second render or later, once its renders have asked for
// this many samples in all) with at most kCacheProbeWalkersPerCu walkers
// per CU times the cached plan the renderer chose against the same launch
// without the cache, and keeps the faster per walker count.  (The cache
// keeps hot cells off the device's atomics but lengthens each walker's
// chain, which bounds renders of few walkers: the Sierpinski triangle at
// 64 walkers per CU rendered faster without it.  With many walkers the
// atomics bound instead: the headline flame's 2048 walkers per CU ran 40
// times slower without the cache, so there is nothing to probe.)
constexpr uint64_t kCacheProbeSamples = 1ull << 28;
constexpr uint64_t kCacheProbeWalkersPerCu = 256;

template <typename R>
static int choose_cache(ffr_renderer *r, const DeviceFlame<R> &d, LaunchPlan &p,
                        uint64_t walker0, uint64_t walkers, uint64_t batch, uint64_t samples)
{
    if (r->cache_pref >= 0 || !p.cache || p.chain || p.bin || p.split_log2)
        return FFR_OK;
    LaunchShape sh = renderer_shape(r);
    sh.cache = 0;
    const auto known = r->cache_choice.find(walkers);
    if (known != r->cache_choice.end()) {
        if (!known->second)
            p = plan_launch(r, walkers, batch, sh);
        return FFR_OK;
    }
    // FFR_CACHE_PROBE_SAMPLES lowers the threshold (tests probe small renders)
    uint64_t threshold = kCacheProbeSamples;
    if (const char *env = std::getenv("FFR_CACHE_PROBE_SAMPLES"))
        threshold = std::strtoull(env, nullptr, 10);
    if (r->launches == 0 || r->samples_asked + samples < threshold ||
        walkers > kCacheProbeWalkersPerCu * (uint64_t)r->cu_count)
        return FFR_OK;
    const LaunchPlan plans[2] = {p, plan_launch(r, walkers, batch, sh)};
    void *const fns[2] = {nullptr, nullptr};
    float ms[2];
    // (one run each when the launch without the cache is far slower)
    const int rc = time_kernels(r, d, plans, fns, 2, walker0, walkers, batch, ms, 1.5f);
    if (rc != FFR_OK)
        return rc;
    // the cache stays unless the launch without it is 3 % faster
    const bool keep = !(ms[1] < 0.97f * ms[0]);
    r->cache_choice[walkers] = keep;
    if (!keep)
        p = plans[1];
    return FFR_OK;
}

// the flame's compiled kernel for this plan (lane-per-walker kernel only),
// compiled on first use; r->rtc_fn stays nullptr when the plan takes
// another kernel, compiled kernels are off, or the probe chose the table
template <typename R>
static int prepare_compiled(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan &p,
                            uint64_t walker0, uint64_t walkers, uint64_t batch, uint64_t last,
                            uint64_t samples)
{
    r->rtc_fn = nullptr;
    if (!r->compiled_pref || p.chain || p.bin || p.split_log2)
        return FFR_OK;
    const int key = (p.cache ? 1 : 0) | (p.block << 1);
    const auto known = r->compiled_choice.find(key);
    const bool probe = r->compiled_pref < 0 && known == r->compiled_choice.end();
    if (r->compiled_pref < 0) {
        if (known != r->compiled_choice.end() && !known->second)
            return FFR_OK;
        // FFR_COMPILED_PROBE_SAMPLES lowers the threshold (tests probe small
        // renders)
        uint64_t threshold = kCompiledProbeSamples;
        if (const char *env = std::getenv("FFR_COMPILED_PROBE_SAMPLES"))
            threshold = std::strtoull(env, nullptr, 10);
        if (probe && (r->launches == 0 || r->samples_asked + samples < threshold))
            return FFR_OK;
    }
    WalkArgs<R> a;
    walk_args(r, d, p, walker0, walkers, batch, last, a);
    RtcKernel k;
    k.mode = r->mode;
    k.dims = r->spec.dims;
    k.nc = walk_nc(r);
    k.vs = r->vs;
    k.cache = p.cache;
    k.block_max = p.cache ? cache_block_max(r->mode == MODE_F64_U64, r->vs) : 256;
    std::string err;
    double compile_s = 0;
    void *fn = nullptr;
    if (rtc_flame_kernel(a, d.cw, k, r->device, &fn, &compile_s, err) != 0)
        return fail(FFR_E_DEVICE, err);
    if (probe) {
        const LaunchPlan plans[2] = {p, p};
        void *const fns[2] = {nullptr, fn};
        float ms[2];
        const int rc = time_kernels(r, d, plans, fns, 2, walker0, walkers, batch, ms);
        if (rc != FFR_OK)
            return rc;
        const bool faster = ms[1] < ms[0];
        r->compiled_choice[key] = faster;
        if (!faster)
            return FFR_OK;
    }
    r->rtc_fn = fn;
    return FFR_OK;
}

template <typename R>
static int launch_single(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan &p,
                         uint64_t walker0, uint64_t walkers, uint64_t batch, uint64_t last)
{
    MissRounds m;
    if (records_wanted(r, p, walkers, batch, (int)sizeof(R)))
        if (const int rc = reserve_records(r, p, walkers, batch, (int)sizeof(R), r->dbuf,
                                           r->miss_tiles, m))
            return rc;
    WalkArgs<R> a[2];
    walk_args(r, d, p, walker0, walkers, batch, last, a[0]);
    records_args(r, p, r->miss_tiles, m, walkers * batch, a);
    r->plain_class = a[0].hot ? -1 : rate_class(walkers * batch);
    r->hargs.resize(sizeof a);
    std::memcpy(r->hargs.data(), a, sizeof a);
    const hipError_t e = hipMemcpyAsync(r->dargs, r->hargs.data(),
                                        m.last ? sizeof a : sizeof a[0], hipMemcpyHostToDevice,
                                        r->stream);
    if (e != hipSuccess)
        return (int)e;
    return launch_rounds<R>(r, p, r->rtc_fn, (int)d.slot_type.size(), r->miss_tiles, m);
}

// walkers and samples per walker of a render of `samples`
static void split_samples(const ffr_renderer *r, uint64_t samples, uint64_t &batch,
                          uint64_t &walkers, uint64_t &last)
{
    batch = r->opt.batch_size ? r->opt.batch_size : ffr_auto_batch(r, samples);
    walkers = (samples + batch - 1) / batch;
    last = samples - (walkers - 1) * batch;
}

// Binned accumulation of one render: passes of `span` iterations of every
// walker (the walkers' points and stream positions carry over in wstate),
// each pass writing at most kBinPassRecords records, sorted by tile and
// added into the buffer before the next pass overwrites them.
template <typename R>
static int launch_binned(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan &p,
                         uint64_t walker0, uint64_t walkers, uint64_t batch, uint64_t last,
                         uint64_t samples)
{
    const uint64_t tw = p.task_walkers;
    const uint64_t slots = (walkers + tw - 1) / tw * tw; // walker slots of the tasks
    // FFR_BIN_PASS_RECORDS makes passes smaller (tests run many passes)
    uint64_t pass_records = kBinPassRecords;
    if (const char *env = std::getenv("FFR_BIN_PASS_RECORDS")) {
        const unsigned long long v = std::strtoull(env, nullptr, 10);
        if (v >= 1 && v < pass_records)
            pass_records = v;
    }
    const uint64_t span = std::max<uint64_t>(1, std::min<uint64_t>(batch, pass_records / slots));
    const uint64_t npass = (batch + span - 1) / span;
    const uint64_t cap = slots * span;
    const int ncol = r->spec.color_dims; // colour components of each record
    hipError_t e =
        r->bin.ensure(BinMemory::sizes(r->cells, ncol, cap, (int)sizeof(R)), cap);
    if (e == hipSuccess && npass > 1)
        e = ensure_device(&r->wstate, r->wstate_bytes, (size_t)slots * sizeof(WalkerState<R>));
    size_t args_bytes = r->dargs_bin_n * sizeof(WalkArgs<R>);
    if (e == hipSuccess)
        e = ensure_device(&r->dargs_bin, args_bytes, (size_t)npass * sizeof(WalkArgs<R>));
    r->dargs_bin_n = args_bytes / sizeof(WalkArgs<R>);
    if (e != hipSuccess)
        return (int)e;
    // one argument block per pass, copied at once (the host copy stays
    // alive until the copy ran)
    r->hargs.resize((size_t)npass * sizeof(WalkArgs<R>));
    for (uint64_t k = 0; k < npass; ++k) {
        WalkArgs<R> a;
        walk_args(r, d, p, walker0, walkers, batch, last, a);
        a.rec = r->bin.b.rec;
        a.wstate = r->wstate;
        a.pay = r->bin.b.pay;
        a.pay_stride = r->bin.b.capacity;
        a.it0 = k * span;
        a.it1 = std::min<uint64_t>(batch, a.it0 + span);
        std::memcpy(r->hargs.data() + k * sizeof a, &a, sizeof a);
    }
    e = hipMemcpyAsync(r->dargs_bin, r->hargs.data(), r->hargs.size(), hipMemcpyHostToDevice,
                       r->stream);
    if (e != hipSuccess)
        return (int)e;
    // The flame's compiled walker (compiled 1; with -1 as for the lane
    // kernel: a renderer in steady use compiles it, and a render of three
    // passes or more times its first pass with the table-driven walker and
    // its second with the compiled one, then keeps the faster for the rest
    // and for later renders).  Both give the same records.
    void *fn = nullptr;
    bool ab = false;
    const int key = 0x100 | (p.block << 9); // (apart from the lane kernel's keys)
    if (r->compiled_pref != 0) {
        const auto known = r->compiled_choice.find(key);
        uint64_t threshold = kCompiledProbeSamples;
        if (const char *env = std::getenv("FFR_COMPILED_PROBE_SAMPLES"))
            threshold = std::strtoull(env, nullptr, 10);
        const bool want =
            r->compiled_pref > 0 || (known != r->compiled_choice.end() && known->second);
        ab = r->compiled_pref < 0 && known == r->compiled_choice.end() && npass >= 3 &&
             r->launches > 0 && r->samples_asked + samples >= threshold;
        if (want || ab) {
            WalkArgs<R> a;
            walk_args(r, d, p, walker0, walkers, batch, last, a);
            RtcKernel k;
            k.mode = r->mode;
            k.dims = r->spec.dims;
            k.nc = walk_nc(r);
            k.vs = r->vs;
            k.block_max = kBinWalkBlock;
            k.bin = true;
            std::string err;
            double compile_s = 0;
            if (rtc_flame_kernel(a, d.cw, k, r->device, &fn, &compile_s, err) != 0)
                return fail(FFR_E_DEVICE, err);
        }
        if (ab)
            for (hipEvent_t &ev : r->ev_ab)
                if (!ev)
                    HIP_TRY(hipEventCreate(&ev));
    }
    void *use = ab ? nullptr : fn;
    for (uint64_t k = 0; k < npass; ++k) {
        // (the walker kernel writes every record of the pass)
        const uint64_t n_rec = slots * (std::min<uint64_t>(batch, (k + 1) * span) - k * span);
        const unsigned char *args = (const unsigned char *)r->dargs_bin + k * sizeof(WalkArgs<R>);
        if (ab && k == 1)
            use = fn;
        if (ab && k < 2)
            HIP_TRY(hipEventRecord(r->ev_ab[2 * k], r->stream));
        int rc;
        if (use) {
            const void *pa = args;
            void *params[] = {&pa};
            rc = (int)hipModuleLaunchKernel((hipFunction_t)use, (unsigned)p.grid, 1, 1,
                                            (unsigned)p.block, 1, 1, (unsigned)p.lds, r->stream,
                                            params, nullptr);
        } else {
            WalkLaunch L;
            L.nc = ncol;
            L.vs = r->vs;
            L.bin = true;
            L.grid = p.grid;
            L.block = p.block;
            L.lds = p.lds;
            L.stream = r->stream;
            L.args = args;
            rc = launch_walk_any(r->mode, r->spec.dims, L);
        }
        if (rc)
            return rc;
        if (ab && k < 2)
            HIP_TRY(hipEventRecord(r->ev_ab[2 * k + 1], r->stream));
        if (ab && k == 1) {
            float t_table = 0, t_compiled = 0;
            HIP_TRY(hipEventSynchronize(r->ev_ab[3]));
            HIP_TRY(hipEventElapsedTime(&t_table, r->ev_ab[0], r->ev_ab[1]));
            HIP_TRY(hipEventElapsedTime(&t_compiled, r->ev_ab[2], r->ev_ab[3]));
            const bool faster = t_compiled < t_table;
            r->compiled_choice[key] = faster;
            use = faster ? fn : nullptr;
            ab = false;
        }
        rc = launch_bin_accumulate(r->bin.b, n_rec, r->cells, r->dbuf, (int)r->word_bytes, ncol,
                                   (int)sizeof(R), r->stream);
        if (rc)
            return rc;
    }
    r->last_compiled = use != nullptr;
    return 0;
}

// records of a split render
static uint64_t split_records(const LaunchPlan &p)
{
    return (uint64_t)p.grid * kSplitBlock * p.split_len;
}

// the scratch of a split render: at most an eighth of the free memory
static hipError_t reserve_split(ffr_renderer *r, const LaunchPlan &p)
{
    const BinMemory n = BinMemory::sizes(r->cells, r->spec.color_dims, split_records(p),
                                         r->mode == MODE_F64_U64 ? 8 : 4);
    BinMemory &mem = r->records.get().split;
    const size_t more = mem.growth(n);
    size_t free_b = 0, total_b = 0;
    if (more && (hipMemGetInfo(&free_b, &total_b) != hipSuccess || more > free_b / 8))
        return hipErrorOutOfMemory;
    const hipError_t e = mem.ensure(n, split_records(p));
    if (e != hipSuccess)
        mem.free_all();
    return e;
}

// A split render: the split walkers write their records, which are binned
// into the buffer; behind them the unsplit kernel of plan `fb`, which runs
// only when the split failed (and then the records are not added).
template <typename R>
static int launch_split_render(ffr_renderer *r, const DeviceFlame<R> &d, const LaunchPlan &p,
                               const LaunchPlan &fb, uint64_t walker0, uint64_t walkers,
                               uint64_t batch, uint64_t last)
{
    WalkArgs<R> a[2];
    walk_args(r, d, fb, walker0, walkers, batch, last, a[0]);
    a[0].split_main = r->dstats;
    a[0].split_xf = r->dxf + r->nxf;
    walk_args(r, d, p, walker0, walkers, batch, last, a[1]);
    a[1].xf_count = r->dxf + r->nxf;
    a[1].split_main = r->dstats;
    a[1].split_len = p.split_len;
    a[1].split_log2 = p.split_log2;
    a[1].split_warm = r->split_warm;
    const BinScratch &bin = r->records.mem->split.b;
    a[1].rec = bin.rec;
    a[1].pay = bin.pay;
    a[1].pay_stride = bin.capacity;
    r->hargs.resize(sizeof a);
    std::memcpy(r->hargs.data(), a, sizeof a);
    hipError_t e = hipMemcpyAsync(r->dargs, r->hargs.data(), sizeof a, hipMemcpyHostToDevice,
                                  r->stream);
    if (e != hipSuccess)
        return (int)e;
    WalkLaunch L;
    L.nc = r->spec.color_dims;
    L.vs = r->vs;
    L.split = true;
    L.grid = p.grid;
    L.block = p.block;
    L.lds = p.lds;
    L.stream = r->stream;
    L.args = (const unsigned char *)r->dargs + sizeof a[0];
    int rc = launch_walk_any(r->mode, r->spec.dims, L);
    if (rc)
        return rc;
    rc = launch_bin_accumulate(bin, split_records(p), r->cells, r->dbuf, (int)r->word_bytes,
                               r->spec.color_dims, (int)sizeof(R), r->stream,
                               &r->dstats->split_fail);
    if (rc)
        return rc;
    return launch_table_kernel(r, fb, (int)d.slot_type.size(), r->dargs);
}

static int launch(ffr_renderer *r, uint64_t samples)
{
    uint64_t batch, walkers, last;
    split_samples(r, samples, batch, walkers, last);
    LaunchPlan p = plan_launch(r, walkers, batch, renderer_shape(r));
    LaunchPlan fb;
    r->last_split = false;
    if (p.split_log2) {
        // (its scratch may be allocated here, so not while the stream is
        // captured; without the memory for it the walkers run unsplit)
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        const bool captured = hipStreamIsCapturing(r->stream, &cap) != hipSuccess ||
                              cap != hipStreamCaptureStatusNone;
        LaunchShape sh = renderer_shape(r);
        sh.split = 0;
        if (!captured && reserve_split(r, p) == hipSuccess) {
            r->last_split = true;
            r->last_split_segments = walkers << p.split_log2;
            sh.bin = 0;
            fb = plan_launch(r, walkers, batch, sh);
        } else {
            (void)hipGetLastError();
            p = plan_launch(r, walkers, batch, sh);
        }
    }
    // (the cache and compiled-kernel probes run first: the reset after them
    // clears what they counted)
    int rc = r->mode == MODE_F64_U64
                 ? choose_cache(r, r->f64, p, r->next_walker, walkers, batch, samples)
                 : choose_cache(r, r->f32, p, r->next_walker, walkers, batch, samples);
    if (rc != FFR_OK)
        return rc;
    r->last_cached = p.cache && !p.direct && !p.bin && !p.split_log2;
    r->last_walkers = walkers;
    r->last_batch = batch;
    r->last_cache = p.cache ? p.slots : 0;
    r->last_chain = p.chain;
    r->last_bin = p.bin;
    rc = r->mode == MODE_F64_U64
             ? prepare_compiled(r, r->f64, p, r->next_walker, walkers, batch, last, samples)
             : prepare_compiled(r, r->f32, p, r->next_walker, walkers, batch, last, samples);
    if (rc != FFR_OK)
        return rc;
    r->last_compiled = r->rtc_fn != nullptr;
    rc = launch_reset_stats(r->dstats, r->dxf, r->nxf, r->stream);
    if (rc)
        return fail(FFR_E_DEVICE, std::string("stats reset: ") + hipGetErrorString((hipError_t)rc));
    if (p.bin || r->last_split) {
        static std::once_flag prepared;
        static int prep_rc = 0;
        std::call_once(prepared, [] { prep_rc = prepare_bin_kernels(); });
        if (prep_rc)
            return fail(FFR_E_DEVICE, std::string("binned accumulation: ") +
                                          hipGetErrorString((hipError_t)prep_rc));
    }
    HIP_TRY(hipEventRecord(r->ev0, r->stream));
    if (r->last_split)
        rc = r->mode == MODE_F64_U64
                 ? launch_split_render(r, r->f64, p, fb, r->next_walker, walkers, batch, last)
                 : launch_split_render(r, r->f32, p, fb, r->next_walker, walkers, batch, last);
    else if (p.bin)
        rc = r->mode == MODE_F64_U64
                 ? launch_binned(r, r->f64, p, r->next_walker, walkers, batch, last, samples)
                 : launch_binned(r, r->f32, p, r->next_walker, walkers, batch, last, samples);
    else
        rc = r->mode == MODE_F64_U64
                 ? launch_single(r, r->f64, p, r->next_walker, walkers, batch, last)
                 : launch_single(r, r->f32, p, r->next_walker, walkers, batch, last);
    if (rc)
        return fail(FFR_E_DEVICE, std::string("walker kernel launch: ") +
                                      hipGetErrorString((hipError_t)rc));
    HIP_TRY(hipEventRecord(r->ev1, r->stream));
    r->next_walker += walkers;
    r->launches += 1;
    r->samples_asked += samples;
    r->pending = true;
    r->timed = true;
    return FFR_OK;
}

static int finish(ffr_renderer *r, ffr_stats *out)
{
    if (r->pending) {
        HIP_TRY(hipStreamSynchronize(r->stream));
        r->pending = false;
        r->records.give_back();
        DevStats st;
        HIP_TRY(hipMemcpy(&st, r->dstats, sizeof st, hipMemcpyDeviceToHost));
        std::vector<unsigned long long> xf((size_t)std::max(r->nxf, 1));
        HIP_TRY(hipMemcpy(xf.data(), r->dxf, sizeof(unsigned long long) * (size_t)r->nxf,
                          hipMemcpyDeviceToHost));
        if (r->timed) {
            float ms = 0;
            HIP_TRY(hipEventElapsedTime(&ms, r->ev0, r->ev1));
            r->last_ms = ms;
        }
        r->s_iter += st.s_iter;
        r->s_plot += st.s_plot;
        for (int k = 0; k < r->nxf; ++k)
            r->xf_dist[(size_t)r->order[(size_t)k]] += xf[(size_t)k];
        for (int i = 0; i < r->spec.dims; ++i) {
            r->pmin[i] = std::min(r->pmin[i], st.pmin[i]);
            r->pmax[i] = std::max(r->pmax[i], st.pmax[i]);
        }
        if (r->last_split) {
            // seams that did not join, or a bad value: unsplit from now on;
            // many segments run twice: a longer run-up
            if (st.split_fail)
                r->split_ok = false;
            else if (st.split_again * 256ull > r->last_split_segments)
                r->split_warm *= 2;
            if (r->split_warm > kSplitWarmMax)
                r->split_ok = false;
            r->last_split = false;
        }
        r->last_bad = st.n_bad;
        if (r->last_cached && st.s_iter) {
            r->miss_rate = (double)(st.atomics - st.flush_atomics) / (double)r->cell_words /
                           (double)st.s_iter;
            if (r->plain_class >= 0)
                r->plain_last = r->plain_rates[r->plain_class] = r->miss_rate;
        }
        r->last_atomics = st.atomics;
        r->last_flush_atomics = st.flush_atomics;
        r->last_records = st.records;
        r->last_pauses = st.pauses;
        // a colour flame whose samples missed the LDS cache often enough
        // renders faster binned from now on
        const double bin_from = miss_ok(r) ? kBinColourRecords : kBinColourAtomics;
        if (r->spec.color_dims > 0 && !r->last_bin && !r->last_chain &&
            st.s_iter >= kBinColourMinSamples &&
            (double)(st.atomics - st.flush_atomics) >= bin_from * (double)st.s_iter)
            r->bin_colour = true;
        size_t nrec = (size_t)std::min<uint64_t>(st.n_bad, r->opt.bad_value_cap);
        r->bv_ids.assign(nrec, 0);
        r->bv_pts.assign(nrec * 3, 0.0);
        if (nrec) {
            HIP_TRY(hipMemcpy(r->bv_ids.data(), r->dbv_xfs, sizeof(uint64_t) * nrec,
                              hipMemcpyDeviceToHost));
            HIP_TRY(hipMemcpy(r->bv_pts.data(), r->dbv_pts, sizeof(double) * 3 * nrec,
                              hipMemcpyDeviceToHost));
            for (auto &id : r->bv_ids)
                id = (uint64_t)r->order[(size_t)id];
        }
    }
    if (out) {
        std::memset(out, 0, sizeof *out);
        out->s_iter = r->s_iter;
        out->s_plot = r->s_plot;
        out->n_bad = r->last_bad;
        out->walkers = r->last_walkers;
        out->batch_size = r->last_batch;
        for (int i = 0; i < 3; ++i) {
            out->pt_min[i] = i < r->spec.dims ? r->pmin[i] : 0.0;
            out->pt_max[i] = i < r->spec.dims ? r->pmax[i] : 0.0;
        }
        out->kernel_ms = r->last_ms;
        out->atomics = r->last_atomics;
        out->flush_atomics = r->last_flush_atomics;
        out->wave_per_walker = r->last_chain ? 1u : 0u;
        out->cache_slots = (uint32_t)r->last_cache;
        out->binned = r->last_bin ? 1u : 0u;
        out->compiled = r->last_compiled ? 1u : 0u;
    }
    if (r->last_bad > r->opt.bad_value_limit)
        return fail(FFR_E_BADVALUE_LIMIT, "render failure (flame may not be sufficiently contractive)");
    return FFR_OK;
}

extern "C" {

int ffr_render_async(ffr_renderer *r, uint64_t samples)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_render_async: null renderer");
    if (r->pending)
        return fail(FFR_E_ARG, "ffr_render_async: a render is already pending (call ffr_sync)");
    HIP_TRY(hipSetDevice(r->device));
    r->bv_ids.clear();
    r->bv_pts.clear();
    r->last_bad = 0;
    if (samples == 0)
        return FFR_OK;
    return launch(r, samples);
}

int ffr_record_use(const ffr_renderer *r, uint64_t *records, uint32_t *pauses)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_record_use: null renderer");
    if (records)
        *records = r->last_records;
    if (pauses)
        *pauses = r->last_pauses;
    return FFR_OK;
}

int ffr_free_idle(int32_t device)
{
    HIP_TRY(hipSetDevice(device));
    (void)RecordPool::of_device(device)->free_idle();
    return FFR_OK;
}

int ffr_sync(ffr_renderer *r, ffr_stats *stats)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_sync: null renderer");
    HIP_TRY(hipSetDevice(r->device));
    return finish(r, stats);
}

int ffr_render(ffr_renderer *r, uint64_t samples, ffr_stats *stats)
{
    int rc = ffr_render_async(r, samples);
    if (rc != FFR_OK)
        return rc;
    return ffr_sync(r, stats);
}

int ffr_set_stream(ffr_renderer *r, void *hip_stream)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_set_stream: null renderer");
    if (r->pending)
        return fail(FFR_E_ARG, "ffr_set_stream: a render is pending");
    if (r->records.mem) { // (of a launch that failed half way)
        HIP_TRY(hipSetDevice(r->device));
        HIP_TRY(hipStreamSynchronize(r->stream));
        r->records.give_back();
    }
    r->stream = hip_stream ? (hipStream_t)hip_stream : r->own_stream;
    return FFR_OK;
}

void *ffr_device_buffer(ffr_renderer *r) { return r ? r->dbuf : nullptr; }
uint64_t ffr_buffer_cells(const ffr_renderer *r) { return r ? r->cells : 0; }
uint32_t ffr_cell_words(const ffr_renderer *r) { return r ? r->cell_words : 0; }
uint32_t ffr_word_bytes(const ffr_renderer *r) { return r ? r->word_bytes : 0; }
size_t ffr_buffer_bytes(const ffr_renderer *r)
{
    return r ? (size_t)r->cells * r->cell_words * r->word_bytes : 0;
}
int32_t ffr_dims(const ffr_renderer *r) { return r ? r->spec.dims : 0; }
int32_t ffr_color_dims(const ffr_renderer *r) { return r ? r->spec.color_dims : 0; }

// memory that the caller pinned
static bool host_pinned(const void *p)
{
    hipPointerAttribute_t at{};
    const bool known = hipPointerGetAttributes(&at, p) == hipSuccess;
    if (!known)
        (void)hipGetLastError();
    return known && at.type != hipMemoryTypeUnregistered;
}

// a copy of a renderer's memory to or from the host, after its stream's work
static hipError_t host_copy(ffr_renderer *r, void *host, void *dev, size_t bytes, bool to_host)
{
    // (a captured stream refuses the wait below, and takes no copies)
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (bytes >= (to_host ? HostStage::kReadBytes : HostStage::kWriteBytes) &&
        hipStreamIsCapturing(r->stream, &cap) == hipSuccess &&
        cap == hipStreamCaptureStatusNone && !host_pinned(host)) {
        HostStage &st = *r->stage;
        std::unique_lock<std::mutex> g(st.busy, std::try_to_lock);
        if (g.owns_lock() && st.wanted(bytes)) {
            if (st.init() == hipSuccess)
                return st.copy(r->device, r->stream, host, dev, bytes, to_host);
            (void)hipGetLastError();
        }
    }
    const hipError_t e = hipStreamSynchronize(r->stream);
    if (e != hipSuccess)
        return e;
    return to_host ? hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost)
                   : hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice);
}

int ffr_read_buffer(ffr_renderer *r, void *dst, size_t bytes)
{
    if (!r || !dst)
        return fail(FFR_E_ARG, "ffr_read_buffer: null argument");
    if (bytes != ffr_buffer_bytes(r))
        return fail(FFR_E_SIZE, "ffr_read_buffer: size mismatch");
    HIP_TRY(hipSetDevice(r->device));
    HIP_TRY(host_copy(r, dst, r->dbuf, bytes, true));
    return FFR_OK;
}

int ffr_write_buffer(ffr_renderer *r, const void *src, size_t bytes)
{
    if (!r || !src)
        return fail(FFR_E_ARG, "ffr_write_buffer: null argument");
    if (bytes != ffr_buffer_bytes(r))
        return fail(FFR_E_SIZE, "ffr_write_buffer: size mismatch");
    HIP_TRY(hipSetDevice(r->device));
    HIP_TRY(host_copy(r, const_cast<void *>(src), r->dbuf, bytes, false));
    return FFR_OK;
}

int ffr_add_buffer(ffr_renderer *r, const void *src, size_t bytes)
{
    if (!r || !src)
        return fail(FFR_E_ARG, "ffr_add_buffer: null argument");
    if (bytes != ffr_buffer_bytes(r))
        return fail(FFR_E_SIZE, "BufferRenderer::addBuffer(): sizes do not match");
    HIP_TRY(hipSetDevice(r->device));
    // staged in chunks of whole cells through one device scratch buffer
    const size_t cell_bytes = (size_t)r->cell_words * r->word_bytes;
    const size_t chunk_cells = std::max<size_t>(1, (size_t)(256u << 20) / cell_bytes);
    const size_t chunk = std::min(bytes, chunk_cells * cell_bytes);
    void *tmp = nullptr;
    HIP_TRY(device_malloc(&tmp, chunk));
    int rc = FFR_OK;
    for (size_t off = 0; off < bytes && rc == FFR_OK; off += chunk) {
        size_t n = std::min(chunk, bytes - off);
        hipError_t e = host_copy(r, (char *)const_cast<void *>(src) + off, tmp, n, false);
        if (e == hipSuccess)
            e = (hipError_t)launch_add_cells((char *)r->dbuf + off, tmp,
                                             n / r->word_bytes, (int)r->cell_words,
                                             (int)r->word_bytes, r->stream);
        if (e == hipSuccess)
            e = hipStreamSynchronize(r->stream);
        if (e != hipSuccess)
            rc = fail(FFR_E_DEVICE, std::string("ffr_add_buffer: ") + hipGetErrorString(e));
    }
    (void)hipFree(tmp);
    return rc;
}

int ffr_add_buffer_noalloc(ffr_renderer *r, const void *src, size_t bytes)
{
    if (!r || !src)
        return fail(FFR_E_ARG, "ffr_add_buffer_noalloc: null argument");
    if (bytes != ffr_buffer_bytes(r))
        return fail(FFR_E_SIZE, "BufferRenderer::addBuffer(): sizes do not match");
    const unsigned long long cell_bytes = (unsigned long long)r->cell_words * r->word_bytes;
    if (cell_bytes > kNoAllocScratchBytes)
        return fail(FFR_E_SIZE, "ffr_add_buffer_noalloc: a cell of " +
                                    std::to_string(cell_bytes) +
                                    " bytes exceeds the staging memory of " +
                                    std::to_string(kNoAllocScratchBytes) + " bytes");
    HIP_TRY(hipSetDevice(r->device));
    const int rc = add_cells_staged_noalloc(r->dbuf, src, bytes, (int)r->cell_words,
                                            (int)r->word_bytes, r->stream);
    if (rc)
        return fail(FFR_E_DEVICE, std::string("ffr_add_buffer_noalloc: ") +
                                      hipGetErrorString((hipError_t)rc));
    return FFR_OK;
}

} // extern "C"

namespace {

// the streamed I/O chunks: 32 MiB of whole cells (or the whole buffer),
// allocated on first use and kept until ffr_destroy
int io_init(ffr_renderer *r)
{
    if (r->io_chunk)
        return FFR_OK;
    const size_t cell_bytes = (size_t)r->cell_words * r->word_bytes;
    const size_t chunk =
        std::min(ffr_buffer_bytes(r), std::max<size_t>(1, (size_t)(32u << 20) / cell_bytes) *
                                          cell_bytes);
    for (int k = 0; k < 2; ++k) {
        HIP_TRY(hipHostMalloc(&r->pin[k], chunk, hipHostMallocDefault));
        HIP_TRY(device_malloc(&r->dchunk[k], chunk));
        HIP_TRY(hipEventCreateWithFlags(&r->io_ev[k], hipEventDisableTiming));
    }
    r->io_chunk = chunk;
    return FFR_OK;
}

// fill dst from the callback until n bytes or the end
size_t read_full(ffr_read_fn read, void *ctx, void *dst, size_t n)
{
    size_t got = 0;
    while (got < n) {
        const size_t k = read(ctx, (char *)dst + got, n - got);
        if (k == 0)
            break;
        got += std::min(k, n - got);
    }
    return got;
}

} // namespace

extern "C" {

int ffr_add_buffer_stream(ffr_renderer *r, ffr_read_fn read, void *ctx)
{
    if (!r || !read)
        return fail(FFR_E_ARG, "ffr_add_buffer_stream: null argument");
    if (r->pending)
        return fail(FFR_E_ARG, "ffr_add_buffer_stream: a render is pending (call ffr_sync)");
    HIP_TRY(hipSetDevice(r->device));
    const int rc0 = io_init(r);
    if (rc0 != FFR_OK)
        return rc0;
    const size_t bytes = ffr_buffer_bytes(r), chunk = r->io_chunk;
    // chunk i goes through pinned buffer i % 2: before it is refilled, the
    // add of chunk i - 2 (which read it through its device chunk) is waited for
    size_t i = 0;
    for (size_t off = 0; off < bytes; off += chunk, ++i) {
        const int k = (int)(i & 1);
        const size_t n = std::min(chunk, bytes - off);
        if (i >= 2)
            HIP_TRY(hipEventSynchronize(r->io_ev[k]));
        if (read_full(read, ctx, r->pin[k], n) != n) {
            HIP_TRY(hipStreamSynchronize(r->stream));
            return fail(FFR_E_IO, "error reading file");
        }
        HIP_TRY(hipMemcpyAsync(r->dchunk[k], r->pin[k], n, hipMemcpyHostToDevice, r->stream));
        HIP_TRY((hipError_t)launch_add_cells((char *)r->dbuf + off, r->dchunk[k],
                                             n / r->word_bytes, (int)r->cell_words,
                                             (int)r->word_bytes, r->stream));
        HIP_TRY(hipEventRecord(r->io_ev[k], r->stream));
    }
    HIP_TRY(hipStreamSynchronize(r->stream));
    return FFR_OK;
}

int ffr_read_buffer_stream(ffr_renderer *r, ffr_write_fn write, void *ctx)
{
    if (!r || !write)
        return fail(FFR_E_ARG, "ffr_read_buffer_stream: null argument");
    if (r->pending)
        return fail(FFR_E_ARG, "ffr_read_buffer_stream: a render is pending (call ffr_sync)");
    HIP_TRY(hipSetDevice(r->device));
    const int rc0 = io_init(r);
    if (rc0 != FFR_OK)
        return rc0;
    const size_t bytes = ffr_buffer_bytes(r), chunk = r->io_chunk;
    const size_t nchunks = (bytes + chunk - 1) / chunk;
    auto issue = [&](size_t i) {
        const int k = (int)(i & 1);
        const size_t off = i * chunk, n = std::min(chunk, bytes - off);
        hipError_t e = hipMemcpyAsync(r->pin[k], (const char *)r->dbuf + off, n,
                                      hipMemcpyDeviceToHost, r->stream);
        if (e == hipSuccess)
            e = hipEventRecord(r->io_ev[k], r->stream);
        return e;
    };
    // the copy of chunk i + 1 runs while chunk i is written out; pinned
    // buffer (i + 1) % 2 held chunk i - 1, which is written out already
    HIP_TRY(issue(0));
    for (size_t i = 0; i < nchunks; ++i) {
        const int k = (int)(i & 1);
        if (i + 1 < nchunks)
            HIP_TRY(issue(i + 1));
        HIP_TRY(hipEventSynchronize(r->io_ev[k]));
        const size_t n = std::min(chunk, bytes - i * chunk);
        if (write(ctx, r->pin[k], n) != n) {
            HIP_TRY(hipStreamSynchronize(r->stream));
            return fail(FFR_E_IO, "error writing output");
        }
    }
    return FFR_OK;
}

int ffr_check_flame(const char *flame_json, size_t len, uint32_t precision, int32_t *ids,
                    double *cw, size_t cap, size_t *n_xforms)
{
    if (!flame_json)
        return fail(FFR_E_ARG, "ffr_check_flame: null flame");
    try {
        Json doc = Json::parse(std::string(flame_json, len));
        FlameSpec spec = parse_flame(doc, precision == FFR_FP32);
        std::vector<int> order;
        std::vector<double> cum;
        if (precision == FFR_FP32) {
            auto d = compile_flame<float>(spec);
            order = d.order;
            for (float v : d.cw)
                cum.push_back((double)v);
        } else {
            auto d = compile_flame<double>(spec);
            order = d.order;
            cum = d.cw;
        }
        for (size_t k = 0; k < order.size() && k < cap; ++k) {
            if (ids)
                ids[k] = order[k];
            if (cw)
                cw[k] = cum[k];
        }
        if (n_xforms)
            *n_xforms = order.size();
    } catch (const std::exception &e) {
        return fail(FFR_E_FLAME, e.what());
    }
    return FFR_OK;
}

int ffr_histogram_l1(ffr_renderer *a, ffr_renderer *b, double *l1)
{
    if (!a || !b || !l1)
        return fail(FFR_E_ARG, "ffr_histogram_l1: null argument");
    if (a->cells != b->cells || a->device != b->device)
        return fail(FFR_E_SIZE, "ffr_histogram_l1: buffers of different shapes or devices");
    uint64_t sa = 0, sb = 0, mn, mx;
    int rc = ffr_histogram_stats(a, &sa, &mn, &mx);
    if (rc)
        return rc;
    rc = ffr_histogram_stats(b, &sb, &mn, &mx);
    if (rc)
        return rc;
    HIP_TRY(hipSetDevice(a->device));
    double *d = reinterpret_cast<double *>(a->dhist); // 3 words of scratch
    HIP_TRY(hipStreamSynchronize(b->stream));
    HIP_TRY((hipError_t)launch_l1_counts(a->dbuf, (int)a->cell_words, (int)a->word_bytes, b->dbuf,
                                         (int)b->cell_words, (int)b->word_bytes, a->cells,
                                         sa ? 1.0 / (double)sa : 0.0, sb ? 1.0 / (double)sb : 0.0,
                                         d, a->stream));
    HIP_TRY(hipMemcpyAsync(l1, d, sizeof(double), hipMemcpyDeviceToHost, a->stream));
    HIP_TRY(hipStreamSynchronize(a->stream));
    return FFR_OK;
}

int ffr_choose_precision(const char *flame_json, size_t len, const ffr_options *opt,
                         uint64_t probe_samples, double threshold, uint32_t *precision,
                         double *l1)
{
    if (!flame_json || !precision)
        return fail(FFR_E_ARG, "ffr_choose_precision: null argument");
    ffr_options o;
    if (opt)
        o = *opt;
    else
        ffr_default_options(&o);
    o.word = FFR_WORD64;
    // both renders draw the same words at the same iteration: one settle
    // count for both (the defaults differ between the precisions)
    if (o.settle_iters < 0)
        o.settle_iters = 53;
    ffr_renderer *r32 = nullptr, *r64 = nullptr;
    o.precision = FFR_FP32;
    int rc = ffr_create(flame_json, len, &o, &r32);
    if (rc == FFR_OK) {
        o.precision = FFR_FP64;
        rc = ffr_create(flame_json, len, &o, &r64);
    }
    int rc32 = FFR_OK, rc64 = FFR_OK;
    if (rc == FFR_OK) {
        rc32 = ffr_render(r32, probe_samples, nullptr);
        rc64 = ffr_render(r64, probe_samples, nullptr);
        if (rc32 != FFR_OK && rc32 != FFR_E_BADVALUE_LIMIT)
            rc = rc32;
        else if (rc64 != FFR_OK && rc64 != FFR_E_BADVALUE_LIMIT)
            rc = rc64;
    }
    double d = 0.0;
    if (rc == FFR_OK)
        rc = ffr_histogram_l1(r32, r64, &d);
    ffr_destroy(r32);
    ffr_destroy(r64);
    if (rc != FFR_OK)
        return rc;
    // an FP32 render stopped by bad values where FP64 was not: the FP32
    // attractor escapes
    const bool escapes = rc32 == FFR_E_BADVALUE_LIMIT && rc64 == FFR_OK;
    *precision = (!escapes && d <= threshold) ? FFR_FP32 : FFR_FP64;
    if (l1)
        *l1 = d;
    return FFR_OK;
}

int ffr_clear_buffer(ffr_renderer *r)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_clear_buffer: null renderer");
    HIP_TRY(hipSetDevice(r->device));
    HIP_TRY((hipError_t)launch_fill_zero(r->dbuf, ffr_buffer_bytes(r), r->stream));
    HIP_TRY(hipStreamSynchronize(r->stream));
    return FFR_OK;
}

int ffr_histogram_stats(ffr_renderer *r, uint64_t *sum, uint64_t *mn, uint64_t *mx)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_histogram_stats: null renderer");
    HIP_TRY(hipSetDevice(r->device));
    HIP_TRY((hipError_t)launch_hist_stats(r->dbuf, r->cells, (int)r->cell_words,
                                          (int)r->word_bytes, r->dhist, r->stream));
    unsigned long long h[3];
    HIP_TRY(hipMemcpyAsync(h, r->dhist, sizeof h, hipMemcpyDeviceToHost, r->stream));
    HIP_TRY(hipStreamSynchronize(r->stream));
    if (sum)
        *sum = h[0];
    if (mn)
        *mn = (r->word_bytes == 4 && h[1] == ~0ull) ? 0xffffffffull : h[1];
    if (mx)
        *mx = h[2];
    return FFR_OK;
}

int ffr_atomic_rate(int32_t device, uint64_t cells, uint32_t cell_words, uint32_t word_bytes,
                    uint64_t updates, double *atomics_per_s)
{
    if (!atomics_per_s || cells == 0 || cells >= (1ull << 32) || cell_words == 0 ||
        cell_words > 5 || (word_bytes != 4 && word_bytes != 8) || updates == 0)
        return fail(FFR_E_ARG, "ffr_atomic_rate: cells in [1, 2^32), 1-5 words of 4 or 8 bytes, "
                               "updates > 0");
    HIP_TRY(hipSetDevice(device));
    const size_t bytes = (size_t)cells * cell_words * word_bytes;
    void *buf = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = FFR_OK;
    float ms = 0.f;
    auto step = [&](hipError_t e, const char *what) {
        if (rc == FFR_OK && e != hipSuccess)
            rc = fail(FFR_E_DEVICE, std::string("ffr_atomic_rate: ") + what + ": " +
                                        hipGetErrorString(e));
        return rc == FFR_OK;
    };
    if (step(device_malloc(&buf, bytes), "hipMalloc") &&
        step(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "stream") &&
        step(hipEventCreate(&e0), "event") && step(hipEventCreate(&e1), "event") &&
        step((hipError_t)launch_fill_zero(buf, bytes, s), "clear") &&
        step((hipError_t)launch_scatter_atomics(buf, cells, (int)cell_words, (int)word_bytes,
                                                std::min<uint64_t>(updates, 1u << 24), s),
             "warm-up") &&
        step(hipEventRecord(e0, s), "record") &&
        step((hipError_t)launch_scatter_atomics(buf, cells, (int)cell_words, (int)word_bytes,
                                                updates, s),
             "scatter") &&
        step(hipEventRecord(e1, s), "record") && step(hipStreamSynchronize(s), "sync") &&
        step(hipEventElapsedTime(&ms, e0, e1), "elapsed")) {
        *atomics_per_s = ms > 0.f ? (double)updates * cell_words / ((double)ms * 1e-3) : 0.0;
    }
    if (e0)
        (void)hipEventDestroy(e0);
    if (e1)
        (void)hipEventDestroy(e1);
    if (s)
        (void)hipStreamDestroy(s);
    (void)hipFree(buf);
    return rc;
}

size_t ffr_image_bytes(const ffr_renderer *r, int mode, int bits)
{
    if (!r || r->spec.dims != 2 || mode < FFR_IMG_MONO || mode > FFR_IMG_COLOR ||
        (bits != 8 && bits != 16))
        return 0;
    const size_t per = mode == FFR_IMG_MONO ? 1 : (size_t)(bits / 8);
    return (size_t)r->cells * (mode == FFR_IMG_COLOR ? 3 : 1) * per;
}

namespace {

// both image entry points: dst is host memory (to_host) or a device address
int render_image(ffr_renderer *r, int mode, double gamma, int bits, void *dst, size_t bytes,
                 ffr_image_info *info, bool to_host)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_render_image: null renderer");
    if (r->pending)
        return fail(FFR_E_ARG, "ffr_render_image: a render is pending (call ffr_sync)");
    // the checks of ffr_img.cpp, in its order (:92-97, :130-134, :149-157,
    // :236-237, :290-291); gamma and the log bound compare against eps of num_t
    const bool f32 = r->word_bytes == 4;
    if (f32 ? (float)gamma < 1e-10f : gamma < 1e-20)
        return fail(FFR_E_ARG, "gamma too small");
    if (bits != 8 && bits != 16)
        return fail(FFR_E_ARG, "bits per channel must be 8 or 16");
    if (r->spec.dims != 2)
        return fail(FFR_E_UNSUPPORTED, "only 2D flames supported");
    if (mode < FFR_IMG_MONO || mode > FFR_IMG_COLOR)
        return fail(FFR_E_ARG,
                    "must choose exactly 1 coloring flag (--monochrome, --grayscale, --color)");
    const size_t need = ffr_image_bytes(r, mode, bits);
    if (dst && (to_host ? bytes != need : bytes < need))
        return fail(FFR_E_SIZE, "ffr_render_image: expected " + std::to_string(need) +
                                    " bytes of pixels");
    HIP_TRY(hipSetDevice(r->device));
    // the pixel kernel takes the bounds from device memory (and writes
    // nothing when the histogram is empty), so one wait covers both passes
    const bool pixels = dst && !(mode == FFR_IMG_COLOR && r->spec.color_dims != 3);
    if (pixels) {
        void *out = dst;
        if (to_host) {
            if (r->dimg_bytes < need) {
                HIP_TRY(hipFree(r->dimg));
                r->dimg = nullptr;
                r->dimg_bytes = 0;
                HIP_TRY(device_malloc(&r->dimg, need));
                r->dimg_bytes = need;
            }
            out = r->dimg;
        }
        HIP_TRY((hipError_t)launch_hist_bounds(r->dbuf, r->cells, (int)r->cell_words,
                                               (int)r->word_bytes, r->dhist, r->stream));
        // num_t gp = 1.0 / arg_gamma (ffr_img.cpp:240): a double division, then num_t
        const double gp = f32 ? (double)(float)(1.0 / (double)(float)gamma) : 1.0 / gamma;
        if (info)
            HIP_TRY(hipEventRecord(r->ev0, r->stream));
        HIP_TRY((hipError_t)launch_tonemap(r->dbuf, r->cells, (int)r->cell_words,
                                           (int)r->word_bytes, mode, r->dhist, gp,
                                           mode == FFR_IMG_MONO ? 8 : bits, out, r->stream));
        if (info)
            HIP_TRY(hipEventRecord(r->ev1, r->stream));
    } else {
        HIP_TRY((hipError_t)launch_hist_stats(r->dbuf, r->cells, (int)r->cell_words,
                                              (int)r->word_bytes, r->dhist, r->stream));
    }
    unsigned long long h[3];
    HIP_TRY(hipMemcpyAsync(h, r->dhist, sizeof h, hipMemcpyDeviceToHost, r->stream));
    HIP_TRY(hipStreamSynchronize(r->stream));
    const uint64_t mn = (f32 && h[1] == ~0ull) ? 0xffffffffull : h[1], mx = h[2];
    // the log scaler's bounds (ffr_img.cpp:223-236), in num_t
    const double smin = f32 ? (double)std::log(1.0f + (float)mn) : std::log(1.0 + (double)mn);
    const double smax = f32 ? (double)std::log(1.0f + (float)mx) : std::log(1.0 + (double)mx);
    if (info) {
        info->hist_min = mn;
        info->hist_max = mx;
        info->scale_min = smin;
        info->scale_max = smax;
        info->width = (uint32_t)r->spec.size[0];
        info->height = (uint32_t)r->spec.size[1];
        info->channels = mode == FFR_IMG_COLOR ? 3u : 1u;
        info->bytes_per_channel = mode == FFR_IMG_MONO ? 1u : (uint32_t)(bits / 8);
        info->kernel_ms = 0.0;
    }
    if (f32 ? (float)smax < 1e-10f : smax < 1e-20)
        return fail(FFR_E_EMPTY, "histogram is (probably) empty");
    if (mode == FFR_IMG_COLOR && r->spec.color_dims != 3)
        return fail(FFR_E_UNSUPPORTED, "buffer must use 3 color dimensions");
    if (!dst)
        return FFR_OK;
    if (to_host)
        HIP_TRY(host_copy(r, dst, r->dimg, need, true));
    if (info) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, r->ev0, r->ev1));
        info->kernel_ms = (double)ms;
    }
    return FFR_OK;
}

} // namespace

int ffr_render_image(ffr_renderer *r, int mode, double gamma, int bits, void *pixels,
                     size_t bytes, ffr_image_info *info)
{
    return render_image(r, mode, gamma, bits, pixels, bytes, info, true);
}

int ffr_render_image_device(ffr_renderer *r, int mode, double gamma, int bits,
                            void *device_pixels, size_t bytes, ffr_image_info *info)
{
    return render_image(r, mode, gamma, bits, device_pixels, bytes, info, false);
}

size_t ffr_xform_id_count(const ffr_renderer *r) { return r ? r->xf_dist.size() : 0; }

int ffr_xform_distribution(const ffr_renderer *r, uint64_t *out, size_t n)
{
    if (!r || (!out && n))
        return fail(FFR_E_ARG, "ffr_xform_distribution: null argument");
    if (n != r->xf_dist.size())
        return fail(FFR_E_SIZE, "ffr_xform_distribution: expected " +
                                    std::to_string(r->xf_dist.size()) + " entries");
    std::copy(r->xf_dist.begin(), r->xf_dist.end(), out);
    return FFR_OK;
}

int ffr_bad_values(const ffr_renderer *r, uint64_t *ids, double *pts, size_t cap, size_t *n)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_bad_values: null renderer");
    size_t m = std::min(cap, r->bv_ids.size());
    const int d = r->spec.dims;
    for (size_t i = 0; i < m; ++i) {
        if (ids)
            ids[i] = r->bv_ids[i];
        if (pts)
            for (int k = 0; k < d; ++k)
                pts[i * (size_t)d + (size_t)k] = r->bv_pts[i * 3 + (size_t)k];
    }
    if (n)
        *n = r->bv_ids.size();
    return FFR_OK;
}

int ffr_xform_order(const ffr_renderer *r, int32_t *ids, double *cw, size_t n)
{
    if (!r)
        return fail(FFR_E_ARG, "ffr_xform_order: null renderer");
    if (n != (size_t)r->nxf)
        return fail(FFR_E_SIZE, "ffr_xform_order: expected " + std::to_string(r->nxf) +
                                    " entries");
    for (int k = 0; k < r->nxf; ++k) {
        if (ids)
            ids[k] = r->order[(size_t)k];
        if (cw)
            cw[k] = r->mode == MODE_F64_U64 ? r->f64.cw[(size_t)k] : (double)r->f32.cw[(size_t)k];
    }
    return FFR_OK;
}

} // extern "C"

#include "ffr_batch.inc"
#include "ffr_server.inc"
