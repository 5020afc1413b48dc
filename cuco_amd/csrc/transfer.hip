// Particle arrays between host and device.
//
// A caller's arrays are pageable and laid out differently from the device's
// (three doubles or a 60-byte record per particle against double4 / float4).
// Copying them whole cost three serial passes over host memory besides the
// link: a zeroed temporary, the runtime's own staging, the repacking loop
// (16777216 particles' positions and velocities: 219 ms for 805 MB).  Here a
// pinned ring of fixed size is filled from one side while the other empties
// it, a slot at a time:
//   down  a kernel packs a slot's particles straight into pinned host memory
//         (no device scratch, no padding over the link), workers move full
//         slots to the caller's array;
//   up    workers fill slots with double4 entries, the copy engine takes
//         them to their place.
// Workers are threads of the call: faulting in the caller's fresh pages is
// most of the host's work and goes about as many times faster as there are
// of them.  Below kInlineDown / kInlineUp bytes no thread is started: six
// cost more than they save (2 MB up: 0.50 ms with them, 0.26 without).
//
// Measured (before -> now, the caller's arrays fresh): positions and
// velocities of 16777216 particles down 219 -> 19 ms (42 GB/s), up 288 -> 33;
// 2097152: down 27.3 -> 3.2, FP32 accelerations 22.6 -> 2.5, records 107 ->
// 3.5, up 36 -> 4.6; 32768: down 0.19 -> 0.09, up 0.27 -> 0.20, FP32
// accelerations 0.049 -> 0.042.  Twelve or sixteen workers are no faster than
// eight.  What does not gain: uploads of some 3000 particles, whose copies
// the runtime takes another way from pinned memory (81 -> 94 us), and their
// FP32 accelerations (14 -> 17 us).  A handle's first large transfer also
// makes the events, and its first round touches the ring.
#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "transfer.h"

namespace cuco {

namespace {

constexpr size_t kSlotBytes = 2u << 20, kMediumSlot = 512u << 10;
constexpr int kWorkers = 8;
constexpr size_t kInlineDown = 2u << 20;

// Component k % 3 of particle k / 3: consecutive lanes write consecutive
// words, and the 16- or 32-byte entries they share come from the cache.
template <typename V, typename T>
__global__ __launch_bounds__(256) void k_pack3(const V *__restrict__ src, uint32_t n,
                                               T *__restrict__ dst)
{
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= 3u * n) return;
    const uint32_t i = k / 3u, c = k - 3u * i;
    const V v = src[i];
    dst[k] = (T)(c == 0u ? v.x : c == 1u ? v.y : v.z);
}

// Word k % 15 of record k / 15 (cuco_particle); rounding to float as the
// host's conversion does.
__global__ __launch_bounds__(256) void k_pack_records(RecordSource s, uint32_t first, uint32_t n,
                                                      uint32_t *__restrict__ dst)
{
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= 15u * n) return;
    const uint32_t r = k / 15u, f = k - 15u * r;
    const uint32_t i = first + r;
    uint32_t out;
    if (f >= 13u) {
        const int32_t *t = f == 13u ? s.ti_end : s.ti_beg;
        out = t ? (uint32_t)t[i] : 0u;
    } else {
        float v;
        if (f < 4u) {
            v = (float)reinterpret_cast<const double *>(s.pos + i)[f];
        } else if (f < 7u) {
            v = (float)reinterpret_cast<const double *>(s.vel + i)[f - 4u];
        } else {
            const bool pp = f < 10u;
            const uint32_t c = pp ? f - 7u : f - 10u;
            const double4 *a64 = pp ? s.pp64 : s.pm64;
            const float4 *a32 = pp ? s.pp32 : s.pm32;
            v = a64   ? (float)reinterpret_cast<const double *>(a64 + i)[c]
                : a32 ? reinterpret_cast<const float *>(a32 + i)[c]
                      : 0.0f;
        }
        out = __float_as_uint(v);
    }
    dst[k] = out;
}

int hip_fail(hipError_t err, const char *what)
{
    set_error("%s failed: %s", what, hipGetErrorString(err));
    return CUCO_ERR_HIP;
}

// The workers of one call: work(k) for k below the published count, in
// order of k; finished(k) tells the publisher when a slot is free again.
class Crew {
public:
    Crew(uint32_t nchunks, int threads, const std::function<void(uint32_t)> &work)
        : work_(work), done_(nchunks, 0)
    {
        threads_.reserve(threads);
        for (int t = 0; t < threads; ++t) {
            try {
                threads_.emplace_back([this] { run(); });
            } catch (const std::exception &) {
                break;  // as many as the system gives; none: the publisher works
            }
        }
    }
    ~Crew() { join(); }
    void publish(uint32_t count)
    {
        if (threads_.empty()) {
            for (; ready_ < count; ++ready_) {
                work_(ready_);
                done_[ready_] = 1;
            }
            return;
        }
        bool several;
        {
            std::lock_guard<std::mutex> g(m_);
            several = count > ready_ + 1u;
            ready_ = count;
        }
        if (several) more_.notify_all();
        else more_.notify_one();
    }
    void wait(uint32_t k)
    {
        std::unique_lock<std::mutex> g(m_);
        freed_.wait(g, [&] { return done_[k] != 0; });
    }
    void join()
    {
        {
            std::lock_guard<std::mutex> g(m_);
            closed_ = true;
        }
        more_.notify_all();
        for (std::thread &t : threads_) t.join();
        threads_.clear();
    }

private:
    void run()
    {
        for (;;) {
            uint32_t k;
            {
                std::unique_lock<std::mutex> g(m_);
                more_.wait(g, [&] { return next_ < ready_ || closed_; });
                if (next_ >= ready_) return;
                k = next_++;
            }
            work_(k);
            {
                std::lock_guard<std::mutex> g(m_);
                done_[k] = 1;
            }
            freed_.notify_all();
        }
    }
    const std::function<void(uint32_t)> &work_;
    std::mutex m_;
    std::condition_variable more_, freed_;
    std::vector<char> done_;
    uint32_t ready_ = 0, next_ = 0;
    bool closed_ = false;
    std::vector<std::thread> threads_;
};

// A thread takes 15-50 us to start: one per 2 MB, as many as pay.
int crew_size(uint32_t nchunks, size_t bytes)
{
    const unsigned hw = std::thread::hardware_concurrency();
    return (int)std::min<uint64_t>({(uint64_t)kWorkers, nchunks, hw ? hw : 1u, bytes / (2u << 20) + 1});
}

}  // namespace

namespace {

// Rings (4 MB at most) that handles have given up, for the next handle: a
// program that makes handles while it holds others would pay a millisecond
// each, as allocating and freeing pinned memory also slows the next device
// allocations.  A ring is idle only after its handle's stream has been
// synchronized; with the last handle all are freed.
struct IdleRing {
    char *pin;
    size_t slot_bytes;
    uint32_t slots;
    int device;
};
constexpr size_t kIdleMost = 4;
std::mutex g_idle_mutex;
std::vector<IdleRing> g_idle;
int g_rings = 0;  // of live handles

}  // namespace

int HostRing::create(uint32_t capacity)
{
    // A handle's ring goes with what it moves: four slots of one FP32 array
    // while that is small (16 KB to 1 MB in all, up to 21845 particles), eight
    // of half a megabyte, or, over a million particles, where the transfers
    // themselves take milliseconds, sixteen of two (of one: 16777216 particles
    // up in 40 ms, not 33).  Default host memory: its first touch takes 8 us
    // a megabyte, that of memory asked to be coherent 375; a slot is read only
    // after an event that releases to the system, or a synchronized stream.
    size_t array = 4096;
    while (array < (size_t)capacity * 12 && array < kMediumSlot) array *= 2;
    const bool large = capacity > 1000000u;
    const size_t want = large ? kSlotBytes : array;
    const uint32_t count = large ? (uint32_t)kSlots : array < kMediumSlot ? 4u : 8u;
    int current = 0;
    const hipError_t de = hipGetDevice(&current);
    if (de != hipSuccess) return hip_fail(de, "hipGetDevice");
    std::lock_guard<std::mutex> guard(g_idle_mutex);
    for (size_t k = 0; k < g_idle.size(); ++k) {
        if (g_idle[k].device != current || g_idle[k].slot_bytes != want || g_idle[k].slots != count)
            continue;
        pin = g_idle[k].pin;
        g_idle.erase(g_idle.begin() + (ptrdiff_t)k);
        break;
    }
    if (!pin) {
        void *p = nullptr;
        if (hipHostMalloc(&p, want * count, hipHostMallocDefault) == hipSuccess) {
            pin = static_cast<char *>(p);
        } else {
            // Pinned memory is not a need of the engine: the transfers only
            // take longer without.
            (void)hipGetLastError();
            pin = static_cast<char *>(std::malloc(want * count));
            const hipError_t err = pin ? hipMalloc(&p, want * count) : hipErrorOutOfMemory;
            if (err != hipSuccess) {
                (void)hipGetLastError();
                std::free(pin);
                pin = nullptr;
                set_error("transfer buffer of %zu bytes refused: %s", want * count,
                          hipGetErrorString(err));
                return CUCO_ERR_OUT_OF_MEMORY;
            }
            dev = static_cast<char *>(p);
        }
    }
    slot_bytes = want;
    slots = count;
    device = current;
    ++g_rings;
    return CUCO_OK;
}

int HostRing::make_events()
{
    for (uint32_t k = 0; k < slots; ++k) {
        if (ev[k]) continue;
        const hipError_t err =
            hipEventCreateWithFlags(&ev[k], hipEventDisableTiming | hipEventReleaseToSystem);
        if (err != hipSuccess) {
            ev[k] = nullptr;
            return hip_fail(err, "hipEventCreate");
        }
    }
    return CUCO_OK;
}

void HostRing::destroy()
{
    for (hipEvent_t &e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (!pin) return;
    std::lock_guard<std::mutex> guard(g_idle_mutex);
    bool kept = false;
    if (dev) {
        (void)hipFree(dev);
        std::free(pin);
        dev = nullptr;
        kept = true;
    } else if (slots < (uint32_t)kSlots && g_idle.size() < kIdleMost) {
        try {
            g_idle.push_back(IdleRing{pin, slot_bytes, slots, device});
            kept = true;
        } catch (const std::exception &) {
        }
    }
    if (!kept) (void)hipHostFree(pin);
    pin = nullptr;
    if (--g_rings == 0) {
        for (const IdleRing &r : g_idle) (void)hipHostFree(r.pin);
        g_idle.clear();
    }
}

int HostRing::pack_slot(uint32_t k, const std::function<int(uint32_t, void *)> &pack,
                        hipStream_t s)
{
    if (!dev) return pack(k, slot(k));
    char *from = dev + (slot(k) - pin);
    const int rc = pack(k, from);
    if (rc) return rc;
    const hipError_t err = hipMemcpyAsync(slot(k), from, slot_bytes, hipMemcpyDeviceToHost, s);
    return err == hipSuccess ? CUCO_OK : hip_fail(err, "hipMemcpyAsync");
}

int HostRing::down(size_t bytes, uint32_t nchunks,
                   const std::function<int(uint32_t, void *)> &pack,
                   const std::function<void(uint32_t, const void *)> &take, hipStream_t s)
{
    std::lock_guard<std::mutex> guard(lock);
    if (nchunks <= slots && bytes <= kInlineDown) {
        for (uint32_t k = 0; k < nchunks; ++k) {
            const int rc = pack_slot(k, pack, s);
            if (rc) {
                (void)hipStreamSynchronize(s);
                return rc;
            }
        }
        const hipError_t err = hipStreamSynchronize(s);
        if (err != hipSuccess) return hip_fail(err, "hipStreamSynchronize");
        for (uint32_t k = 0; k < nchunks; ++k) take(k, slot(k));
        return CUCO_OK;
    }
    int rc = make_events();
    if (rc) return rc;
    const std::function<void(uint32_t)> work = [&](uint32_t k) { take(k, slot(k)); };
    Crew crew(nchunks, crew_size(nchunks, bytes), work);
    // Slot k is packed while up to ahead slots before it are still on their
    // way and the older ones are being emptied.
    const uint32_t ahead = slots / 2;
    uint32_t launched = 0;
    for (uint32_t k = 0; k < nchunks + ahead && !rc; ++k) {
        if (k < nchunks) {
            if (k >= slots) crew.wait(k - slots);
            rc = pack_slot(k, pack, s);
            if (rc) break;
            const hipError_t err = hipEventRecord(ev[k % slots], s);
            if (err != hipSuccess) {
                rc = hip_fail(err, "hipEventRecord");
                break;
            }
            launched = k + 1;
        }
        if (k >= ahead && k - ahead < launched) {
            const hipError_t err = hipEventSynchronize(ev[(k - ahead) % slots]);
            if (err != hipSuccess) {
                rc = hip_fail(err, "hipEventSynchronize");
                break;
            }
            crew.publish(k - ahead + 1);
        }
    }
    crew.join();
    if (rc) (void)hipStreamSynchronize(s);
    return rc;
}

int HostRing::up(size_t bytes, uint32_t nchunks, uint32_t held,
                 const std::function<void(uint32_t, void *)> &fill,
                 const std::function<int()> &ready,
                 const std::function<int(uint32_t, const void *)> &send, hipStream_t s)
{
    std::lock_guard<std::mutex> guard(lock);
    int rc = CUCO_OK;
    if (bytes <= kInlineUp) {
        for (uint32_t k = 0; k < held; ++k) fill(k, slot(k));
        rc = ready();
        if (rc) return rc;
        for (uint32_t k = 0; k < held && !rc; ++k) rc = send(k, slot(k));
        for (uint32_t k = held; k < nchunks && !rc; ++k) {
            if (k && k % slots == 0) {  // the slots are free again
                const hipError_t err = hipStreamSynchronize(s);
                if (err != hipSuccess) {
                    rc = hip_fail(err, "hipStreamSynchronize");
                    break;
                }
            }
            fill(k, slot(k));
            rc = send(k, slot(k));
        }
    } else {
        rc = make_events();
        if (rc) return rc;
        const std::function<void(uint32_t)> work = [&](uint32_t k) { fill(k, slot(k)); };
        Crew crew(nchunks, crew_size(nchunks, bytes), work);
        crew.publish(held);
        for (uint32_t k = 0; k < held; ++k) crew.wait(k);
        rc = ready();
        uint32_t open = held;  // chunks the workers may fill
        for (uint32_t k = 0; k < nchunks && !rc; ++k) {
            // A slot is free again when the copy out of it has ended.
            const uint32_t want = std::min(nchunks, k + slots / 2);
            for (; open < want && !rc; ++open) {
                if (open >= slots) {
                    const hipError_t err = hipEventSynchronize(ev[open % slots]);
                    if (err != hipSuccess) rc = hip_fail(err, "hipEventSynchronize");
                }
                if (!rc) crew.publish(open + 1);
            }
            if (rc) break;
            crew.wait(k);
            rc = send(k, slot(k));
            if (rc) break;
            const hipError_t err = hipEventRecord(ev[k % slots], s);
            if (err != hipSuccess) rc = hip_fail(err, "hipEventRecord");
        }
        crew.join();
    }
    const hipError_t err = hipStreamSynchronize(s);
    if (!rc && err != hipSuccess) rc = hip_fail(err, "hipStreamSynchronize");
    return rc;
}

void for_chunks(size_t bytes, uint32_t nchunks, const std::function<void(uint32_t)> &work)
{
    if (bytes <= kInlineUp) {
        for (uint32_t k = 0; k < nchunks; ++k) work(k);
        return;
    }
    Crew crew(nchunks, crew_size(nchunks, bytes), work);
    crew.publish(nchunks);
    crew.join();
}

int launch_pack3(const double4 *src, uint32_t n, double *dst, hipStream_t s)
{
    k_pack3<<<(3u * n + 255u) / 256u, 256, 0, s>>>(src, n, dst);
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

int launch_pack3(const double4 *src, uint32_t n, float *dst, hipStream_t s)
{
    k_pack3<<<(3u * n + 255u) / 256u, 256, 0, s>>>(src, n, dst);
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

int launch_pack3(const float4 *src, uint32_t n, float *dst, hipStream_t s)
{
    k_pack3<<<(3u * n + 255u) / 256u, 256, 0, s>>>(src, n, dst);
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

int launch_pack_records(const RecordSource &src, uint32_t first, uint32_t n, void *dst,
                        hipStream_t s)
{
    k_pack_records<<<(15u * n + 255u) / 256u, 256, 0, s>>>(src, first, n,
                                                           static_cast<uint32_t *>(dst));
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

}  // namespace cuco
