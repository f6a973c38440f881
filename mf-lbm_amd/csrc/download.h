// Downloads of padded device fields into the caller's arrays in the reference's halo layouts.
//
// A kernel packs the halo box of a field into pinned host memory in the caller's element order, a chunk at a time
// through a ring of RING buffers, while up to MAX_THREADS host threads copy the chunks that have arrived into the
// caller's (pageable, often never touched) array.  Copying whole padded arrays into a pageable buffer and unpacking
// them row by row on one thread was bound by page faults and that thread: 139 ms for the five fields of a 256^3
// lattice (0.70 GB, 5 GB/s), 26 ms so (27 GB/s).
#pragma once
#include <hip/hip_runtime.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "device_common.h"

namespace mflbm_dev {

// one array to download: value e of dst is the S value at src[stride * padded offset], widened to double, over the box
// of halo h
struct DownloadItem {
    const void* src;
    int f32;      // the source is float
    int stride;
    int h;
    double* dst;
};

static __global__ void __launch_bounds__(BLOCK) k_pack_box(Layout L, DownloadItem it, long first, int count, double* out) {
    const int t = (int)blockIdx.x * BLOCK + (int)threadIdx.x;
    if (t >= count) return;
    const long e = first + t;
    const int sx = L.nx + 2 * it.h, sy = L.ny + 2 * it.h;
    const long row = e / sx;
    const int i = (int)(e - row * sx) + 1 - it.h, j = (int)(row % sy) + 1 - it.h, k = (int)(row / sy) + 1 - it.h;
    const long o = (long)it.stride * L.at(i, j, k);
    out[t] = it.f32 ? (double)((const float*)it.src)[o] : ((const double*)it.src)[o];
}

class Downloader {
    static constexpr int RING = 4, MAX_THREADS = 8;
    static constexpr long CHUNK = 1L << 19;   // doubles (4 MiB): a chunk is on the bus for about 0.1 ms
    double* ring = nullptr;                   // pinned, kept with the context; at most RING * CHUNK doubles
    long ring_chunk = 0;                      // doubles per buffer
    hipEvent_t ev[RING] = {};

   public:
    void free() {
        if (ring) (void)hipHostFree(ring);
        ring = nullptr;
        ring_chunk = 0;
        for (hipEvent_t& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    // the items in turn, after the work already on the stream; returns when every dst is written.  Small downloads take
    // the calling thread alone.
    hipError_t run(const Layout& L, hipStream_t stream, const std::vector<DownloadItem>& items) {
        struct Chunk {
            int item;
            long first;
            int count;
        };
        long most = 0, total = 0;
        for (const DownloadItem& it : items) {
            const long n = (long)(L.nx + 2 * it.h) * (L.ny + 2 * it.h) * (L.nz + 2 * it.h);
            most = std::max(most, n);
            total += n;
        }
        if (total == 0) return hipStreamSynchronize(stream);
        const long size = std::min(most, CHUNK);
        hipError_t e = hipSuccess;
        if (size > ring_chunk) {
            if (ring) (void)hipHostFree(ring);
            ring = nullptr;
            ring_chunk = 0;
            if ((e = hipHostMalloc((void**)&ring, sizeof(double) * RING * size)) != hipSuccess) return e;
            ring_chunk = size;
        }
        for (hipEvent_t& v : ev)
            if (!v && (e = hipEventCreateWithFlags(&v, hipEventDisableTiming | hipEventReleaseToSystem)) != hipSuccess) return e;
        std::vector<Chunk> chunks;
        for (size_t m = 0; m < items.size(); ++m) {
            const int h = items[m].h;
            const long n = (long)(L.nx + 2 * h) * (L.ny + 2 * h) * (L.nz + 2 * h);
            for (long f = 0; f < n; f += ring_chunk) chunks.push_back(Chunk{(int)m, f, (int)std::min(ring_chunk, n - f)});
        }
        const int nc = (int)chunks.size();
        int nt = 1;
        if (total > CHUNK) {
            cpu_set_t set;
            const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
            nt = std::max(1, std::min(MAX_THREADS, cpus));
        }
        // chunk c is in buffer c % RING; `arrived` chunks are there, and a buffer is filled again when `copied` of its
        // chunk says that every thread has taken its part
        std::atomic<int> arrived{0};
        std::vector<std::atomic<int>> copied(nc);
        for (auto& a : copied) a.store(0, std::memory_order_relaxed);
        auto part = [&](int c, int t, int of) {
            const Chunk& k = chunks[c];
            const long a = (long)k.count * t / of, b = (long)k.count * (t + 1) / of;
            std::memcpy(items[k.item].dst + k.first + a, ring + (c % RING) * ring_chunk + a, sizeof(double) * (b - a));
            copied[c].fetch_add(1, std::memory_order_release);
        };
        std::atomic<int> team{0};   // threads the parts are cut for; 0 until they are started
        std::vector<std::thread> threads;
        auto worker = [&](int t) {
            int of;
            while ((of = team.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
            for (int c = 0; c < nc; ++c) {
                int a;
                while ((a = arrived.load(std::memory_order_acquire)) <= c) {
                    if (a < 0) return;   // the device failed
                    std::this_thread::yield();
                }
                part(c, t, of);
            }
        };
        int of = 1, launched = 0;
        for (int c = 0; c < nc && e == hipSuccess; ++c) {
            for (; launched < nc && launched < c + RING && e == hipSuccess; ++launched) {
                if (launched >= RING)
                    while (copied[launched - RING].load(std::memory_order_acquire) < of) std::this_thread::yield();
                const Chunk& k = chunks[launched];
                hipLaunchKernelGGL(k_pack_box, dim3(nblocks(k.count)), dim3(BLOCK), 0, stream, L, items[k.item], k.first,
                                   k.count, ring + (launched % RING) * ring_chunk);
                if ((e = hipGetLastError()) == hipSuccess) e = hipEventRecord(ev[launched % RING], stream);
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev[c % RING]);
            if (e != hipSuccess) break;
            if (c == 0 && nt > 1) {   // the work queued before the download is done: now the threads have something to do
                try {
                    threads.reserve(nt - 1);
                    for (int t = 1; t < nt; ++t) threads.emplace_back(worker, t);
                } catch (const std::exception&) {   // fewer threads than asked for: the parts are cut for those there are
                }
                of = (int)threads.size() + 1;
                team.store(of, std::memory_order_release);
            }
            arrived.store(c + 1, std::memory_order_release);
            part(c, 0, of);
        }
        if (e != hipSuccess) arrived.store(-1, std::memory_order_release);
        for (std::thread& t : threads) t.join();
        return e;
    }
};

}  // namespace mflbm_dev
