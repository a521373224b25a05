// hostio.hip -- large host CSR arrays to and from device matrices through a
// ring of pinned staging slots.
//
// A copy from or to pageable memory runs through the runtime's own staging on
// one host thread, and moves 64-bit indices that the device then narrows
// (widens).  Here a team of host threads narrows columns and offsets to 32
// bits while it fills (widens them while it empties) the slots, the calling
// thread queues a copy kernel per slot, and the two overlap; pages of a freshly
// allocated output are first touched by the team, too.  Bytes over the bus: 12
// instead of 16 per nonzero.  The bus bounds it: 56 GB/s in one large copy of
// pinned memory, 37 here, 36 in and 18 out for pageable memory.  Drop-in product
// of a 7-point 80^3 operator (162 MB of host arrays, 0.2 ms of it the product):
// 7.0 ms with pageable copies, 3.9 this way.  Copies by the DMA engines instead
// of the kernel (a gap behind each): 4.6 ms.
#include <sched.h>

#include <atomic>
#include <memory>
#include <thread>

#include "engine.hpp"

namespace sp3mm {

namespace {
constexpr size_t kSlotBytes = (size_t)1 << 20;
constexpr int kSlots = 16;
constexpr int kGroup = 4;  // copies per event
constexpr int kTeam = 6;  // threads beside the caller at most (4: 4.0 ms, 5 to 8: 3.9, 12: 4.2)

enum class Kind { Raw, Cols, Offsets };

// one run of elements of an array: `h` on the host (64-bit for Cols and
// Offsets), `d` on the device (32-bit for those)
struct Chunk {
    Kind kind;
    unsigned char *h, *d;
    size_t n, bytes;  // elements, bytes on the device
    int64_t first;    // index of the first element in its array
};

void cut(std::vector<Chunk> &out, Kind kind, const void *h, void *d, size_t n, size_t hsize, size_t dsize)
{
    const size_t per = kSlotBytes / dsize;
    auto *hb = static_cast<unsigned char *>(const_cast<void *>(h));
    auto *db = static_cast<unsigned char *>(d);
    for (size_t i = 0; i < n; i += per) {
        const size_t m = std::min(per, n - i);
        out.push_back(Chunk{kind, hb + i * hsize, db + i * dsize, m, m * dsize, (int64_t)i});
    }
}

int team_size()
{
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    return std::min(kTeam, cpus - 1);
}

inline void relax(unsigned &spins)
{
    if ((++spins & 255) == 0) sched_yield();
    else __builtin_ia32_pause();
}

// The state a team shares.  Slot j % kSlots belongs to chunk j; `open` is the
// number of chunks whose slots the threads may use, and ready[j] is set once
// chunk j has been filled (emptied).
struct Team {
    const std::vector<Chunk> &ch;
    std::unique_ptr<std::atomic<char>[]> ready;
    std::atomic<int> next{0}, open{0};
    std::atomic<bool> stop{false};
    std::vector<std::thread> threads;

    explicit Team(const std::vector<Chunk> &c) : ch(c), ready(new std::atomic<char>[c.size()]())
    {
        threads.reserve(kTeam);
    }
    ~Team()
    {
        stop = true;
        join();
    }
    void join()
    {
        for (auto &t : threads) t.join();
        threads.clear();
    }
    template <typename Work>
    bool start(int n, Work work)
    {
        for (int k = 0; k < n; k++) {
            try {
                threads.emplace_back([this, work] {
                    for (;;) {
                        const int j = next.fetch_add(1);
                        if (j >= (int)ch.size()) return;
                        for (unsigned spins = 0; j >= open.load(std::memory_order_acquire); relax(spins))
                            if (stop.load(std::memory_order_relaxed)) return;
                        work(j);
                        ready[j].store(1, std::memory_order_release);
                    }
                });
            } catch (...) {
                break;  // fewer threads
            }
        }
        return !threads.empty();
    }
};

// Copies a slot over the bus.  16 workgroups have enough bytes in flight for
// it (80^3 drop-in product: 4 workgroups 4.4 ms, 8 and 16 3.9, 64 and 256 4.1).
__global__ void __launch_bounds__(256) k_bus_copy(uint4 *__restrict__ d, const uint4 *__restrict__ s, int n, int tail)
{
    const int step = gridDim.x * 256;
    int i = blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.x == 0 && (int)threadIdx.x < tail)
        reinterpret_cast<uint32_t *>(d + n)[threadIdx.x] = reinterpret_cast<const uint32_t *>(s + n)[threadIdx.x];
    for (; i + 3 * step < n; i += 4 * step) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = s[i + u * step];
#pragma unroll
        for (int u = 0; u < 4; u++) d[i + u * step] = v[u];
    }
    for (; i < n; i += step) d[i] = s[i];
}

// bytes: a multiple of 4; both sides 16-byte aligned (slots, and multiples of
// a slot's size into allocations)
hipError_t bus_copy(void *d, const void *s, size_t bytes, hipStream_t st)
{
    hipLaunchKernelGGL(k_bus_copy, dim3(16), dim3(256), 0, st, static_cast<uint4 *>(d), static_cast<const uint4 *>(s),
                       (int)(bytes / 16), (int)(bytes % 16 / 4));
    return hipGetLastError();
}

bool aligned16(const sp3mm_dmat &m)
{
    return ((reinterpret_cast<uintptr_t>(m.rp32) | reinterpret_cast<uintptr_t>(m.col) |
             reinterpret_cast<uintptr_t>(m.val)) & 15) == 0;
}

void drop_ring(HostRing *r)
{
    for (auto e : r->ev) (void)hipEventDestroy(e);
    if (r->mem) (void)hipHostFree(r->mem);
    delete r;
}

bool ring_ready(Context *c)
{
    if (c->ring) return true;
    auto *r = new (std::nothrow) HostRing();
    if (!r) return false;
    bool ok = hipHostMalloc((void **)&r->mem, kSlotBytes * kSlots, hipHostMallocCoherent | hipHostMallocMapped) ==
                  hipSuccess &&
              hipHostGetDevicePointer((void **)&r->dev, r->mem, 0) == hipSuccess;
    for (int i = 0; ok && i < kSlots / kGroup; i++) {
        hipEvent_t e;
        ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        if (ok) r->ev.push_back(e);
    }
    if (!ok) {
        (void)hipGetLastError();
        drop_ring(r);
        return false;
    }
    c->ring = r;
    return true;
}

// Below this many bytes of host arrays the threads' start costs what the faster
// copies give back (7-point drop-in products: 40^3, 4 to 8 MB per operand, 1.04
// ms this way and 1.02 pageable; 48^3, 7 to 13 MB, 1.26 and 1.63).
constexpr size_t kMinBytes = (size_t)6 << 20;
}  // namespace

// under the context's lock, behind its stream
void ring_release(Context *c)
{
    if (c->ring) drop_ring(c->ring);
    c->ring = nullptr;
}

// memory the runtime knows nothing of, which it would stage itself
static bool pageable(const void *p)
{
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

// Arrays in pinned memory are not staged: one copy of each runs at the bus's
// rate, and the pages of a new array are not touched from the host.  7-point
// operators, up / down in ms: 48^3 0.32 / 0.28 against 0.41 / 0.34 staged, 96^3
// 2.15 / 1.91 against 2.15 / 1.80, and into new pinned arrays 1.9 against 9 to 12.
bool host_io_fits(int64_t M, int64_t nnz, int vtype, const int64_t *ja, const void *val)
{
    return nnz < INT32_MAX &&
           (size_t)(M + 1) * 8 + (size_t)nnz * (8 + (vtype == SP3MM_F32 ? 4 : 8)) >= kMinBytes &&
           (pageable(ja) || pageable(val));
}

int host_upload(Context *c, const sp3mm_dmat &m, const int64_t *irp, const int64_t *ja, const void *val, int base,
                HostCheck &chk)
{
    const int n = team_size();
    if (n < 2 || !aligned16(m) || !ring_ready(c)) return 1;
    const size_t vs = m.vtype == SP3MM_F32 ? 4 : 8;
    std::vector<Chunk> ch;
    std::atomic<int64_t> bad_row{INT64_MAX};
    std::atomic<bool> bad_col{false};
    std::unique_ptr<Team> team;  // joined before what its threads use goes
    try {
        cut(ch, Kind::Offsets, irp, m.rp32, (size_t)m.M + 1, 8, 4);
        cut(ch, Kind::Cols, ja, m.col, (size_t)m.nnz, 8, 4);
        cut(ch, Kind::Raw, val, m.val, (size_t)m.nnz, vs, vs);
        team.reset(new Team(ch));
    } catch (...) {
        return 1;
    }
    unsigned char *mem = c->ring->mem;
    const int64_t last = m.N - 1, M = m.M;
    auto fill = [&, mem, last, M, base](int j) {
        const Chunk &k = ch[(size_t)j];
        void *slot = mem + (size_t)(j % kSlots) * kSlotBytes;
        if (k.kind == Kind::Raw) {
            __builtin_memcpy(slot, k.h, k.bytes);
            return;
        }
        const auto *src = reinterpret_cast<const uint64_t *>(k.h);
        auto *dst = static_cast<int32_t *>(slot);
        for (size_t i = 0; i < k.n; i++) dst[i] = (int32_t)(uint32_t)(src[i] - (uint64_t)base);
        if (k.kind == Kind::Cols) {
            uint64_t out = 0;  // sign bit: a column below 0 or above `last`
            for (size_t i = 0; i < k.n; i++) {
                const uint64_t v = src[i] - (uint64_t)base;
                out |= v | ((uint64_t)last - v);
            }
            if (out >> 63) bad_col = true;
        } else {
            const auto *off = reinterpret_cast<const int64_t *>(k.h);
            bool down = false;
            const size_t pairs = (size_t)std::min<int64_t>((int64_t)k.n, M - k.first);
            for (size_t i = 0; i < pairs; i++) down |= off[i + 1] < off[i];
            for (size_t i = 0; down && i < pairs; i++)
                if (off[i + 1] < off[i]) {
                    const int64_t r = k.first + (int64_t)i;
                    for (int64_t was = bad_row.load(); r < was && !bad_row.compare_exchange_weak(was, r);) {
                    }
                    break;
                }
        }
    };
    team->open = kSlots;
    if (!team->start(n, fill)) return 1;
    hipError_t e = hipSuccess;
    const int total = (int)ch.size();
    int queued = 0, done = 0;
    for (unsigned spins = 0; queued < total && e == hipSuccess;) {
        if (team->ready[queued].load(std::memory_order_acquire)) {
            const Chunk &k = ch[(size_t)queued];
            const int slot = queued % kSlots;
            e = bus_copy(k.d, c->ring->dev + (size_t)slot * kSlotBytes, k.bytes, c->stream);
            if (e == hipSuccess && ++queued % kGroup == 0) e = hipEventRecord(c->ring->ev[slot / kGroup], c->stream);
        } else if (done + kGroup <= queued) {
            const hipError_t q = hipEventQuery(c->ring->ev[done % kSlots / kGroup]);
            if (q == hipSuccess) team->open.store((done += kGroup) + kSlots, std::memory_order_release);
            else if (q != hipErrorNotReady) e = q;
        } else {
            relax(spins);
        }
    }
    if (e != hipSuccess) team->stop = true;
    team->join();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);  // no copy may still read the ring
        set_error("upload: HIP error %s", hipGetErrorString(e));
        return -1;
    }
    chk.bad_row = bad_row == INT64_MAX ? -1 : bad_row.load();
    chk.bad_col = bad_col;
    return 0;
}

int host_download(Context *c, const sp3mm_dmat &m, int64_t *irp, int64_t *ja, void *val, int base)
{
    const int n = team_size();
    if (n < 2 || !m.rp32 || !aligned16(m) || !ring_ready(c)) return 1;
    const size_t vs = m.vtype == SP3MM_F32 ? 4 : 8;
    std::vector<Chunk> ch;
    std::unique_ptr<Team> team;
    try {
        cut(ch, Kind::Offsets, irp, m.rp32, (size_t)m.M + 1, 8, 4);
        if (ja) cut(ch, Kind::Cols, ja, m.col, (size_t)m.nnz, 8, 4);
        if (val) cut(ch, Kind::Raw, val, m.val, (size_t)m.nnz, vs, vs);
        team.reset(new Team(ch));
    } catch (...) {
        return 1;
    }
    unsigned char *mem = c->ring->mem;
    auto empty = [&, mem, base](int j) {
        const Chunk &k = ch[(size_t)j];
        const void *slot = mem + (size_t)(j % kSlots) * kSlotBytes;
        if (k.kind == Kind::Raw) {
            __builtin_memcpy(k.h, slot, k.bytes);
            return;
        }
        auto *dst = reinterpret_cast<int64_t *>(k.h);
        const auto *src = static_cast<const int32_t *>(slot);
        for (size_t i = 0; i < k.n; i++) dst[i] = (int64_t)src[i] + base;
    };
    if (!team->start(n, empty)) return 1;
    hipError_t e = hipSuccess;
    const int total = (int)ch.size();
    int queued = 0, here = 0;
    for (unsigned spins = 0; here < total && e == hipSuccess;) {
        if (queued < total &&
            (queued < kSlots || team->ready[queued - kSlots].load(std::memory_order_acquire))) {
            const Chunk &k = ch[(size_t)queued];
            const int slot = queued % kSlots;
            e = bus_copy(c->ring->dev + (size_t)slot * kSlotBytes, k.d, k.bytes, c->stream);
            queued++;
            if (e == hipSuccess && (queued % kGroup == 0 || queued == total))
                e = hipEventRecord(c->ring->ev[slot / kGroup], c->stream);
        } else if (here < queued) {
            // a whole group is queued, or the last chunks are: its slots were
            // free together or free up without what is waited for here
            const int upto = std::min(here / kGroup * kGroup + kGroup, total);
            const hipError_t q = upto <= queued ? hipEventQuery(c->ring->ev[here % kSlots / kGroup]) : hipErrorNotReady;
            if (q == hipSuccess) team->open.store(here = upto, std::memory_order_release);
            else if (q != hipErrorNotReady) e = q;
        } else {
            relax(spins);
        }
    }
    if (e != hipSuccess) team->stop = true;
    team->join();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);
        set_error("download: HIP error %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}

}  // namespace sp3mm
