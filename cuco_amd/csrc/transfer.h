// Ring between a caller's arrays and the device (transfer.hip): pinned host
// memory, or, where the system gives none, ordinary memory and as much of the
// device's.
#pragma once

#include <functional>
#include <mutex>

#include "internal.h"

namespace cuco {

struct HostRing {
    static constexpr int kSlots = 16;  // at most
    char *pin = nullptr;
    // Where pinned memory is refused, pin is ordinary memory and the device
    // packs into these slots, which are copied down.
    char *dev = nullptr;
    size_t slot_bytes = 0;
    uint32_t slots = 0;
    int device = 0;
    hipEvent_t ev[kSlots] = {};  // made by the first transfer that needs them
    std::mutex lock;  // one transfer of a handle at a time

    int create(uint32_t capacity);
    int make_events();
    void destroy();
    char *slot(uint32_t k) { return pin + (size_t)(k % slots) * slot_bytes; }
    // pack, and the copy down where the ring is not pinned.
    int pack_slot(uint32_t k, const std::function<int(uint32_t, void *)> &pack, hipStream_t s);
    // Entries of `size` bytes in a slot.
    uint32_t entries(size_t size) const { return (uint32_t)(slot_bytes / size); }

    // Chunks 0..nchunks-1 (bytes in all): pack launches the work that fills
    // a slot, take empties it (any thread; must not throw or use HIP).
    int down(size_t bytes, uint32_t nchunks, const std::function<int(uint32_t, void *)> &pack,
             const std::function<void(uint32_t, const void *)> &take, hipStream_t s);
    // fill fills a slot (any thread, likewise), send launches its copy; ends
    // with the stream synchronized.  The first held chunks (at most as many as
    // slots) are all filled before ready is called, and nothing is sent where
    // that returns an error.
    int up(size_t bytes, uint32_t nchunks, uint32_t held,
           const std::function<void(uint32_t, void *)> &fill, const std::function<int()> &ready,
           const std::function<int(uint32_t, const void *)> &send, hipStream_t s);
};

// Most bytes an upload takes without threads.
constexpr size_t kInlineUp = 4u << 20;

// work(0..nchunks-1), on several threads where it reads enough bytes.
void for_chunks(size_t bytes, uint32_t nchunks, const std::function<void(uint32_t)> &work);

// x, y, z of n entries, packed.
int launch_pack3(const double4 *src, uint32_t n, double *dst, hipStream_t s);
int launch_pack3(const double4 *src, uint32_t n, float *dst, hipStream_t s);
int launch_pack3(const float4 *src, uint32_t n, float *dst, hipStream_t s);

// What cuco_particle records are made of; null: zeros.
struct RecordSource {
    const double4 *pos = nullptr, *vel = nullptr;
    const double4 *pp64 = nullptr, *pm64 = nullptr;
    const float4 *pp32 = nullptr, *pm32 = nullptr;
    const int32_t *ti_end = nullptr, *ti_beg = nullptr;
};
int launch_pack_records(const RecordSource &src, uint32_t first, uint32_t n, void *dst,
                        hipStream_t s);

}  // namespace cuco
