// The transfer ring (transfer.hip, host side) against a HIP runtime made of
// threads: a stream runs its operations in order on a thread of its own, some
// of them late, so that a slot that is read before its event, or filled again
// before it is free, shows as wrong bytes.  Prints "ok" when all cases hold.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "transfer.h"

namespace {

struct Stream {
    std::mutex m;
    std::condition_variable cv;
    std::deque<std::function<void()>> q;
    uint64_t put = 0, done = 0;
    bool stop = false;
    std::thread t{[this] { run(); }};
    void run()
    {
        for (;;) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> g(m);
                cv.wait(g, [&] { return stop || !q.empty(); });
                if (q.empty()) return;
                f = std::move(q.front());
                q.pop_front();
            }
            f();
            {
                std::lock_guard<std::mutex> g(m);
                ++done;
            }
            cv.notify_all();
        }
    }
    void add(std::function<void()> f)
    {
        {
            std::lock_guard<std::mutex> g(m);
            q.push_back(std::move(f));
            ++put;
        }
        cv.notify_all();
    }
    uint64_t mark()
    {
        std::lock_guard<std::mutex> g(m);
        return put;
    }
    void wait(uint64_t upto)
    {
        std::unique_lock<std::mutex> g(m);
        cv.wait(g, [&] { return done >= upto; });
    }
    ~Stream()
    {
        {
            std::lock_guard<std::mutex> g(m);
            stop = true;
        }
        cv.notify_all();
        t.join();
    }
};

struct Event {
    Stream *s = nullptr;
    uint64_t at = 0;
};

std::mutex g_m;
std::map<void *, size_t> g_pinned, g_device;
int g_pin_calls = 0;
bool g_refuse_pinned = false, g_refuse_device = false;
std::atomic<int> g_events{0};
int g_failures = 0;

#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);     \
            ++g_failures;                                           \
        }                                                           \
    } while (0)

void late(uint32_t k)
{
    if (k % 3 == 1) std::this_thread::sleep_for(std::chrono::microseconds(300));
}

}  // namespace

// ------------------------------------------------------------ the runtime
extern "C" {
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> g(g_m);
    ++g_pin_calls;
    if (g_refuse_pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    g_pinned[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::lock_guard<std::mutex> g(g_m);
    CHECK(g_pinned.erase(p) == 1);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> g(g_m);
    if (g_refuse_device) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    g_device[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> g(g_m);
    CHECK(g_device.erase(p) == 1);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t s)
{
    reinterpret_cast<Stream *>(s)->add([=] { std::memcpy(to, from, n); });
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    ++g_events;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    --g_events;
    delete reinterpret_cast<Event *>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    Event *ev = reinterpret_cast<Event *>(e);
    ev->s = reinterpret_cast<Stream *>(s);
    ev->at = ev->s->mark();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    Event *ev = reinterpret_cast<Event *>(e);
    if (ev->s) ev->s->wait(ev->at);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    Stream *st = reinterpret_cast<Stream *>(s);
    st->wait(st->mark());
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}
}

namespace cuco {
void set_error(const char *, ...) {}
}  // namespace cuco

// ------------------------------------------------------------ the cases
namespace {

using cuco::HostRing;

uint64_t word(uint32_t k, size_t i) { return k * 1000003ull + i * 7ull + 1ull; }

// nchunks chunks of a whole slot down; bytes: what the ring is told.
void check_down(HostRing &r, Stream &s, uint32_t nchunks, size_t bytes, int fail_at = -1)
{
    const size_t n = r.slot_bytes / 8;
    std::vector<std::atomic<int>> seen(nchunks);
    for (auto &x : seen) x = 0;
    std::atomic<int> wrong{0};
    const int rc = r.down(
        bytes, nchunks,
        [&](uint32_t k, void *slot) {
            if ((int)k == fail_at) return 7;
            s.add([=] {
                late(k);
                for (size_t i = 0; i < n; ++i) static_cast<uint64_t *>(slot)[i] = word(k, i);
            });
            return 0;
        },
        [&](uint32_t k, const void *slot) {
            if (k % 7 == 2) std::this_thread::sleep_for(std::chrono::milliseconds(3));
            const uint64_t *v = static_cast<const uint64_t *>(slot);
            for (size_t i = 0; i < n; i += 17) wrong += v[i] != word(k, i);
            wrong += v[n - 1] != word(k, n - 1);
            ++seen[k];
        },
        reinterpret_cast<hipStream_t>(&s));
    CHECK(rc == (fail_at < 0 ? 0 : 7));
    CHECK(wrong == 0);
    for (uint32_t k = 0; k < nchunks; ++k) CHECK(fail_at >= 0 ? seen[k] <= 1 : seen[k] == 1);
}

void check_up(HostRing &r, Stream &s, uint32_t nchunks, uint32_t held, size_t bytes,
              bool refuse = false, int fail_at = -1)
{
    const size_t n = r.slot_bytes / 8;
    std::vector<std::atomic<int>> filled(nchunks), got(nchunks);
    for (auto &x : filled) x = 0;
    for (auto &x : got) x = 0;
    std::atomic<int> wrong{0}, sent{0};
    bool asked = false;
    const int rc = r.up(
        bytes, nchunks, held,
        [&](uint32_t k, void *slot) {
            late(k + 2);
            for (size_t i = 0; i < n; ++i) static_cast<uint64_t *>(slot)[i] = word(k, i);
            ++filled[k];
        },
        [&]() -> int {
            asked = true;
            CHECK(sent == 0);
            for (uint32_t k = 0; k < held; ++k) CHECK(filled[k] == 1);
            return refuse ? 9 : 0;
        },
        [&](uint32_t k, const void *slot) {
            CHECK(filled[k] == 1);
            ++sent;
            if ((int)k == fail_at) return 7;
            s.add([&, k, slot] {
                late(k);
                const uint64_t *v = static_cast<const uint64_t *>(slot);
                for (size_t i = 0; i < n; i += 13) wrong += v[i] != word(k, i);
                wrong += v[n - 1] != word(k, n - 1);
                ++got[k];
            });
            return 0;
        },
        reinterpret_cast<hipStream_t>(&s));
    CHECK(asked);
    CHECK(rc == (refuse ? 9 : fail_at >= 0 ? 7 : 0));
    CHECK(wrong == 0);
    if (refuse) CHECK(sent == 0);
    if (!refuse && fail_at < 0)
        for (uint32_t k = 0; k < nchunks; ++k) CHECK(got[k] == 1);
}

void check_ring(HostRing &r, Stream &s)
{
    const uint32_t S = r.slots;
    const size_t small = 1000, large = 64u << 20;
    for (uint32_t n : {1u, 2u, S - 1, S, S + 1, 2 * S, 2 * S + 3, 5 * S + 1}) {
        for (size_t bytes : {small, large}) {
            check_down(r, s, n, bytes);
            for (uint32_t held : {0u, 1u, std::min(n, S)}) {
                check_up(r, s, n, held, bytes);
                check_up(r, s, n, held, bytes, true);
            }
        }
        check_down(r, s, n, large, (int)n / 2);
        check_up(r, s, n, 0, large, false, (int)n / 2);
        check_up(r, s, n, std::min(n, S), small, false, (int)n - 1);
    }
    check_down(r, s, 0, 0);
    check_down(r, s, 3, small);
}

}  // namespace

int main()
{
    // Sizes on either side of the ring's kinds, pinned or not.
    for (bool refuse : {false, true}) {
        g_refuse_pinned = refuse;
        for (uint32_t cap : {1u, 341u, 342u, 21845u, 21846u, 1000000u, 1000001u}) {
            Stream s;
            HostRing r;
            CHECK(r.create(cap) == 0);
            CHECK((r.dev != nullptr) == refuse);
            CHECK(r.slot_bytes * r.slots >= std::min<size_t>((size_t)cap * 32, 4u << 20));
            if (cap < 1000001u) check_ring(r, s);
            else {
                check_down(r, s, 2 * r.slots + 1, 64u << 20);
                check_up(r, s, 2 * r.slots + 1, r.slots, 64u << 20);
            }
            r.destroy();
            CHECK(g_pinned.empty() && g_device.empty() && g_events == 0);
        }
    }
    // Neither pinned nor device memory: an error, and nothing held.
    g_refuse_device = true;
    {
        HostRing r;
        CHECK(r.create(1000) == CUCO_ERR_OUT_OF_MEMORY);
        r.destroy();
    }
    g_refuse_pinned = g_refuse_device = false;

    // Rings that handles leave: taken by the next of the same size while
    // another lives, not by one of another size; all freed with the last.
    {
        Stream s;
        HostRing keep, a, b, c;
        CHECK(keep.create(50000) == 0 && a.create(5000) == 0);
        check_ring(a, s);
        char *was = a.pin;
        const int calls = g_pin_calls;
        a.destroy();
        CHECK(b.create(500) == 0 && b.pin != was && g_pin_calls == calls + 1);
        CHECK(c.create(5000) == 0 && c.pin == was && g_pin_calls == calls + 1);
        check_ring(c, s);
        // Six more closed: four stay.
        {
            HostRing more[6];
            for (HostRing &m : more) CHECK(m.create(2000000 / 100) == 0);
            const size_t live = g_pinned.size();
            for (HostRing &m : more) m.destroy();
            CHECK(g_pinned.size() == live - 2);
        }
        b.destroy();
        c.destroy();
        CHECK(g_pinned.size() == 5);
        keep.destroy();
        CHECK(g_pinned.empty() && g_events == 0);
    }

    // Two handles on two threads, and two threads on one handle.
    {
        Stream s0, s1;
        HostRing r0, r1;
        CHECK(r0.create(32768) == 0 && r1.create(1000001) == 0);
        std::thread a([&] { check_ring(r0, s0); });
        std::thread b([&] {
            for (int k = 0; k < 3; ++k) check_down(r1, s1, 20, 64u << 20);
        });
        std::thread c([&] {
            for (int k = 0; k < 3; ++k) check_up(r1, s1, 20, 16, 64u << 20);
        });
        a.join();
        b.join();
        c.join();
        r0.destroy();
        r1.destroy();
    }
    CHECK(g_pinned.empty() && g_device.empty() && g_events == 0);
    if (g_failures == 0) std::printf("ok\n");
    return g_failures != 0;
}
