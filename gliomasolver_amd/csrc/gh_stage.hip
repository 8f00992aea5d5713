// gh_stage.hip -- fields between the device and the caller's memory.
//
// The caller's arrays are pageable and often fresh: a copy into them is bound by
// page faults and by one core's memcpy (17 GB/s into fresh pages, 55 GB/s over
// the bus on MI355X), and a dense array was put together from block-major order
// on the host in a buffer of its own size.  Here a kernel writes the caller's
// order into pinned slabs, and up to four threads move the slabs, two each, so
// that one is filled while the other is emptied.  A field of 256^3 FP32 cells
// arrives in 2.4 ms (21 before), 128^3 in 0.3 ms (0.75), 32^3 in 25 us (60).
//
// The slabs outlive a call: eight of 512 KiB and eight of 128 KiB at most per
// device, shared by every context and thread under a mutex, freed with the last
// context.  Pinning
// costs 0.5 ms a MiB, which a program that moves one field must win back, so the
// slabs are small (of 2 MiB they save another 0.4 ms at 256^3 and cost 6 ms
// once), and transfers within 128 KiB take smaller ones.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "gh_ctx.h"
#include "gh_slab_pool.h"

namespace gh {
namespace {

constexpr size_t kSlabBytes = 512u << 10;
constexpr size_t kSmallSlab = 128u << 10;
constexpr int kStageThreads = 4;
constexpr size_t kThreadedBytes = 1u << 20;  // 60 us of copying; starting three threads takes 30

struct Slab {
    void* p = nullptr;
    size_t bytes = 0;
    hipEvent_t ev = nullptr;  // recorded after the slab's last use on the device
    int device = 0;
};

std::mutex g_mu;
SlabPool<Slab> g_free;
int g_users = 0;

void drop(Slab& s) {
    if (s.ev) (void)hipEventDestroy(s.ev);
    if (s.p) (void)hipHostFree(s.p);
    s = Slab{};
}

// a slab of at least `need` bytes
int take(int device, size_t need, Slab& s) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_free.take(device, need, s)) return GH_OK;
    }
    s.device = device;
    s.bytes = need <= kSmallSlab ? kSmallSlab : kSlabBytes;
    GH_HIP_CHECK(hipHostMalloc(&s.p, s.bytes, hipHostMallocDefault));
    GH_HIP_CHECK(hipEventCreateWithFlags(&s.ev, hipEventDisableTiming));
    return GH_OK;
}

// a slab no device work uses any more
void give(Slab& s) {
    if (!s.p && !s.ev) return;
    try {
        std::lock_guard<std::mutex> lock(g_mu);
        if (s.p && s.ev && g_users > 0 && g_free.give(s)) {
            s = Slab{};
            return;
        }
    } catch (...) {  // no memory for the list
    }
    drop(s);
}

// a thread's slabs (one where one chunk is all it moves); given back when the
// device is done with them, freed (which waits for the device) after a failure
struct Pair {
    Slab s[2];
    bool used[2] = {false, false};
    bool whole = false;
    int take_for(int device, size_t bytes) {
        int rc = take(device, std::min(bytes, kSlabBytes), s[0]);
        return rc || bytes <= kSlabBytes ? rc : take(device, kSlabBytes, s[1]);
    }
    int finish() {
        for (int i = 0; i < 2; ++i)
            if (used[i]) GH_HIP_CHECK(hipEventSynchronize(s[i].ev));
        whole = true;
        return GH_OK;
    }
    ~Pair() {
        for (int i = 0; i < 2; ++i) whole ? give(s[i]) : drop(s[i]);
    }
};

// Threads for a transfer of n chunks: one, and one more for each pair of slabs that
// lies ready.  So a transfer pins two slabs at most (0.5 ms), a program that moves
// one field pays for no more, and the fourth transfer has its four threads.
int threads_for(int device, size_t n) {
    std::lock_guard<std::mutex> lock(g_mu);
    return (int)std::min<size_t>({(size_t)kStageThreads, n, 1 + g_free.ready(device, kSlabBytes) / 2});
}

// Runs part(first, last) over the chunks of `bytes` on up to kStageThreads
// threads; the first failure's code and message.
template <typename F>
int in_parts(int device, size_t bytes, F part) {
    const size_t n = (bytes + kSlabBytes - 1) / kSlabBytes;
    const int nt = bytes < kThreadedBytes ? 1 : threads_for(device, n);
    if (nt <= 1) return part((size_t)0, n);
    int rc[kStageThreads] = {};
    std::string msg[kStageThreads];
    auto run = [&](int t) {
        rc[t] = part(n * t / nt, n * (t + 1) / nt);
        try {
            if (rc[t]) msg[t] = last_error();
        } catch (...) {
        }
    };
    std::thread th[kStageThreads];
    int started = 1;
    try {
        for (; started < nt; ++started) th[started] = std::thread(run, started);
    } catch (...) {  // no more threads: the rest runs here
    }
    run(0);
    for (int t = started; t < nt; ++t) run(t);
    for (int t = 1; t < started; ++t) th[t].join();
    for (int t = 0; t < nt; ++t)
        if (rc[t]) return set_error(rc[t], msg[t]);
    return GH_OK;
}

// device -> dst: fill(offset, bytes, slab) enqueues a chunk of the result
template <typename Fill>
int fetch(int device, hipStream_t stream, size_t bytes, void* dst, Fill fill) {
    return in_parts(device, bytes, [&](size_t c0, size_t c1) -> int {
        GH_HIP_CHECK(hipSetDevice(device));
        auto size = [&](size_t c) { return std::min(kSlabBytes, bytes - c * kSlabBytes); };
        Pair p;
        int rc;
        if ((rc = p.take_for(device, std::min(bytes, (c1 - c0) * kSlabBytes)))) return rc;
        for (size_t c = c0; c <= c1; ++c) {  // chunk c is filled while chunk c - 1 is emptied
            if (c < c1) {
                Slab& s = p.s[(c - c0) & 1];
                if ((rc = fill(c * kSlabBytes, size(c), s.p))) return rc;
                GH_HIP_CHECK(hipEventRecord(s.ev, stream));
            }
            if (c > c0) {
                Slab& s = p.s[(c - 1 - c0) & 1];
                GH_HIP_CHECK(hipEventSynchronize(s.ev));
                std::memcpy((char*)dst + (c - 1) * kSlabBytes, s.p, size(c - 1));
            }
        }
        return p.finish();
    });
}

// src -> device: drain(offset, bytes, slab) enqueues a chunk's use
template <typename Drain>
int send(int device, hipStream_t stream, size_t bytes, const void* src, Drain drain) {
    return in_parts(device, bytes, [&](size_t c0, size_t c1) -> int {
        GH_HIP_CHECK(hipSetDevice(device));
        Pair p;
        int rc;
        if ((rc = p.take_for(device, std::min(bytes, (c1 - c0) * kSlabBytes)))) return rc;
        for (size_t c = c0; c < c1; ++c) {
            const int i = (int)((c - c0) & 1);
            Slab& s = p.s[i];
            if (p.used[i]) GH_HIP_CHECK(hipEventSynchronize(s.ev));
            const size_t o = c * kSlabBytes, n = std::min(kSlabBytes, bytes - o);
            std::memcpy(s.p, (const char*)src + o, n);
            if ((rc = drain(o, n, s.p))) return rc;
            GH_HIP_CHECK(hipEventRecord(s.ev, stream));
            p.used[i] = true;
        }
        return p.finish();
    });
}

struct alignas(16) Unit {
    unsigned w[4];
};

// `units` 16-byte units of a field, from unit `first` of the caller's order on,
// between the block-major field and a slab, consecutive lanes on consecutive units
// of the slab.  UPR: units to a row of a block where the caller's order is the
// dense x-fastest one of a uniform grid (slots bx + bpd * (by + bpd * bz)), 0 where
// it is block-major too.  A kernel's stores cross the bus at the rate of a copy
// engine and start 20 us sooner (3 MB of an adaptive grid: 230 -> 80 us).
template <int UPR, bool FETCH>
__global__ __launch_bounds__(256) void units_kernel(int bpd, size_t first, unsigned units, Unit* f, Unit* slab) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= units) return;
    Unit* b = f + first + i;
    if constexpr (UPR > 0) {
        const unsigned n = BS * bpd, row = UPR * bpd, u = (unsigned)first + i;  // below 2^27: n <= 512
        const unsigned ux = u % row, yz = u / row, y = yz % n, z = yz / n;
        const size_t s = ux / UPR + (size_t)bpd * ((y >> 3) + (size_t)bpd * (z >> 3));
        b = f + (s * 64 + (y & 7) + 8 * (z & 7)) * UPR + ux % UPR;
    }
    if (FETCH)
        slab[i] = *b;
    else
        *b = slab[i];
}

// bpd 0: block-major (a fetch only)
template <bool FETCH>
int units(hipStream_t stream, int bpd, size_t real_size, void* f, size_t offset, size_t bytes, void* slab) {
    const unsigned n = (unsigned)(bytes / 16);
    auto* k = real_size == 4 ? units_kernel<2, FETCH> : units_kernel<4, FETCH>;
    if constexpr (FETCH)
        if (bpd == 0) k = units_kernel<0, true>;
    hipLaunchKernelGGL(k, dim3((n + 255) / 256), dim3(256), 0, stream, bpd, offset / 16, n, (Unit*)f, (Unit*)slab);
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

}  // namespace

void stage_retain() {
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_users;
}
void stage_release() {
    std::vector<Slab> gone;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_users == 0) gone.swap(g_free.slabs);
    }
    for (Slab& s : gone) drop(s);
}

int stage_fetch(int device, hipStream_t stream, const void* field, size_t cells, int bpd, size_t real_size, void* dst) {
    return fetch(device, stream, cells * real_size, dst, [&](size_t o, size_t n, void* slab) {
        return units<true>(stream, bpd, real_size, const_cast<void*>(field), o, n, slab);
    });
}

int stage_send(int device, hipStream_t stream, void* field, size_t cells, int bpd, size_t real_size, const void* src) {
    return send(device, stream, cells * real_size, src, [&](size_t o, size_t n, void* slab) {
        return units<false>(stream, bpd, real_size, field, o, n, slab);
    });
}

}  // namespace gh
