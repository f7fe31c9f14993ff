// Reading device data into the caller's (pageable) arrays.
//
// A copy of device memory to pageable memory goes through the runtime's own
// staging, one piece after the other: 17 GB/s on MI355X.  Here the kernel that
// puts the values into the caller's layout writes them straight into pinned
// host memory, piece by piece, and up to three threads take finished pieces on
// to the caller's array while the next ones are written: 48 GB/s for 400 MB
// (27 with one thread; a conversion into device memory followed by a copy of
// each piece 35; pieces of 1, 2 and 4 MB 45, 48 and 50), with no device staging.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <string>
#include <thread>

#include "fastdiv.hpp"
#include "state.hpp"

namespace plb {

// The pinned pieces of one state or batch: allocated by its first read (for
// that read and for the velocities of as many cells, and again for a larger
// one: at most 12 MB), freed with it.  Two pieces per thread that such a read
// takes: one being written, one being read.
// One read at a time holds them; reads of one state or batch from several
// threads wait for each other.
struct HostRing {
    static constexpr int kThreads = 3;
    static constexpr int kSlots = 2 * kThreads;
    static constexpr size_t kSlotBytes = (size_t)2 << 20;  // largest piece
    char* buf = nullptr;
    size_t slot_bytes = 0;
    int slots = 0;
    hipEvent_t ev[kSlots] = {};
    std::mutex held;
};

inline void host_ring_free(HostRing* r) {
    for (hipEvent_t& e : r->ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (r->buf) (void)hipHostFree(r->buf);
    r->buf = nullptr;
}

inline int host_ring_ensure(HostRing* r, size_t slot_bytes, int slots) {
    for (int i = 0; i < slots; ++i)
        if (!r->ev[i]) PLB_HIP_TRY(hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming));
    if (r->buf && r->slot_bytes >= slot_bytes && r->slots >= slots) return PLB_OK;
    if (r->buf) PLB_HIP_TRY(hipHostFree(r->buf));
    r->buf = nullptr;
    size_t size = std::max(r->slot_bytes, (size_t)64 << 10);
    while (size < slot_bytes) size *= 2;
    slots = std::max(slots, r->slots);
    void* p = nullptr;
    PLB_HIP_TRY(hipHostMalloc(&p, slots * size, hipHostMallocDefault));
    r->buf = (char*)p;
    r->slot_bytes = size;
    r->slots = slots;
    return PLB_OK;
}

// Threads of a read: they pay for themselves from about 4 MB on.
inline int host_read_threads(uint64_t bytes) {
    return (int)std::min<uint64_t>(HostRing::kThreads, 1 + bytes / (4u << 20));
}

// Reads `items` items of item_bytes each: fill(first, count, slot) launches on
// the stream the kernel that writes items [first, first + count) to the pinned
// slot; put(first, count, slot) takes them from there to the caller's array
// (items of different pieces concurrently).  Pieces are handed out in order,
// whichever threads could be started.
template <class Fill, class Put>
int host_read(HostRing* r, int device, hipStream_t stream, uint64_t items, size_t item_bytes, const Fill& fill,
              const Put& put) {
    if (items == 0) return PLB_OK;
    // pieces of an eighth of what is read, so that writing and taking overlap in
    // a small read too, but no less than 512 KB: each costs a launch and a wait
    // (1.1 MB in pieces of 128, 256 and 512 KB: 88, 64 and 58 us; 2.2 MB 115, 118 and 102)
    const uint64_t most = HostRing::kSlotBytes / item_bytes,
                   least = std::max<uint64_t>(1, std::min<uint64_t>(most, (512u << 10) / item_bytes));
    const uint64_t piece = std::min(items, std::max(least, std::min(most, (items + 7) / 8)));
    const uint64_t pieces = (items + piece - 1) / piece;
    std::lock_guard<std::mutex> hold(r->held);
    // not once for a density and again for the velocities (24 bytes a cell)
    // that are read after it: setting pinned memory up again costs 2 ms
    const uint64_t cells = std::min(items, std::max<uint64_t>((512u << 10) / 24,
                                                             std::min<uint64_t>(HostRing::kSlotBytes / 24, (items + 7) / 8)));
    const uint64_t larger = std::max<uint64_t>(items * item_bytes, items * 24);
    const int rc = host_ring_ensure(r, std::max<size_t>(piece * item_bytes, cells * 24), 2 * host_read_threads(larger));
    if (rc) return rc;
    const size_t slot_bytes = r->slot_bytes;
    std::atomic<uint64_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int w) {
        hipError_t e = hipSetDevice(device);
        uint64_t held = 0, count = 0;  // the piece in flight, count = 0: none
        for (int i = 0; e == hipSuccess; i ^= 1) {
            const uint64_t p = failed.load() == (int)hipSuccess ? next.fetch_add(1) : pieces;
            const int slot = 2 * w + i;
            uint64_t n = 0;
            if (p < pieces) {
                n = std::min(piece, items - p * piece);
                e = fill(p * piece, n, r->buf + slot * slot_bytes);
                if (e == hipSuccess) e = hipEventRecord(r->ev[slot], stream);
            }
            if (count && e == hipSuccess) {
                const int s = 2 * w + (i ^ 1);
                e = hipEventSynchronize(r->ev[s]);
                if (e == hipSuccess) put(held, count, r->buf + s * slot_bytes);
            }
            if (n == 0) break;
            held = p * piece;
            count = n;
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    const int threads = host_read_threads(items * item_bytes);
    std::thread others[HostRing::kThreads];
    for (int w = 1; w < threads; ++w) {
        try {
            others[w] = std::thread(work, w);
        } catch (const std::exception&) {
            break;  // the threads there are do the rest
        }
    }
    work(0);
    for (std::thread& t : others)
        if (t.joinable()) t.join();
    if (failed.load() != (int)hipSuccess) {
        // nothing may go on writing the slots after a failed read
        (void)hipStreamSynchronize(stream);
        return fail(PLB_ERR_HIP, std::string("download: ") + hipGetErrorString((hipError_t)failed.load()));
    }
    return PLB_OK;
}

// The kernel of a read: consecutive values (cell after cell, vlen values each)
// from get(cell, v), in 16-byte stores (the bus takes whole lines).
template <class H, class Get>
__global__ void k_host_fill(Get get, uint64_t first, uint32_t values, FastDiv dv, H* __restrict__ out) {
    constexpr uint32_t W = 16 / sizeof(H);
    typedef H HV __attribute__((ext_vector_type(W)));
    for (uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * W; i < values; i += gridDim.x * blockDim.x * W) {
        HV o;
#pragma unroll
        for (uint32_t j = 0; j < W; ++j) {
            const uint32_t t = std::min(i + j, values - 1u), c = fdiv(t, dv);
            o[j] = (H)get(first + c, t - c * dv.d);
        }
        if (i + W <= values) {
            *reinterpret_cast<HV*>(out + i) = o;
        } else {
            for (uint32_t j = 0; i + j < values; ++j) out[i + j] = o[j];
        }
    }
}

template <class H, class Get>
hipError_t host_fill(const Get& get, uint64_t first, uint64_t cells, int vlen, void* slot, hipStream_t stream) {
    const uint32_t values = (uint32_t)(cells * (uint64_t)vlen);  // at most a slot of them
    constexpr uint32_t W = 16 / sizeof(H);
    const uint32_t blocks = std::min(512u, (values + 256u * W - 1u) / (256u * W));
    hipLaunchKernelGGL((k_host_fill<H, Get>), dim3(blocks), dim3(256), 0, stream, get, first, values,
                       make_fastdiv((uint32_t)vlen), (H*)slot);
    return hipGetLastError();
}

// Interior cells to the caller's halo'd array (the reference's layout), row
// piece by row piece; its halo stays as it is.
inline void put_rows(void* host, const void* slot, uint64_t first, uint64_t count, size_t cell_bytes, uint64_t X,
                     uint64_t Y) {
    const char* from = (const char*)slot;
    for (uint64_t c = first; c < first + count;) {
        const uint64_t x = c % X, row = c / X, y = row % Y, z = row / Y;
        const uint64_t n = std::min(X - x, first + count - c);
        const uint64_t to = ((z + 1) * (Y + 2) + y + 1) * (X + 2) + x + 1;
        std::memcpy((char*)host + to * cell_bytes, from, n * cell_bytes);
        from += n * cell_bytes;
        c += n;
    }
}

}  // namespace plb
