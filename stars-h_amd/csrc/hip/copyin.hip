// Upload of many host arrays into one device buffer (the factors and dense
// tiles of a compressed matrix, for products and the error measure).
//
// The arrays are packed into a ring of pinned slots by several host threads
// while earlier slots are on their way to the device, so that the transfer
// runs at the rate of the bus.  Packing them into one ordinary buffer with one
// thread first, and letting the runtime stage that, took 95 ms for the 430 MB
// of a 64000-point operator: page faults of the buffer, the copy, and a
// transfer through the runtime's own staging.  This takes 9.7 ms, 44 GB/s
// with the allocation, and 69 ms for the 3.4 GB of a 65536-point Matern
// operator.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>
#include "hip_common.h"

namespace {

constexpr int64_t CHUNK = (int64_t)1 << 21;     // doubles per slot: 16 MiB
constexpr int NSLOT = 8;
constexpr int64_t PIECE = (int64_t)1 << 16;     // doubles per copy: 512 KiB
// below this the threads cost more than they save: an operator of 5.4 MB is
// built in 0.31 ms without them and 0.33 with, one of 10.8 MB in 0.54 and 0.37
constexpr int64_t SMALL = (int64_t)1 << 20;     // doubles: 8 MiB

// The ring, kept between calls (as many slots as the largest upload took, at
// most 128 MiB); one upload uses it at a time.  A second one at the same time,
// or one that gets no pinned memory or no thread, takes the simple path.
std::mutex ring_mu;
double *ring = nullptr;
int64_t ring_slots = 0;
hipEvent_t ring_ev[NSLOT] = {};

// False (and no HIP error left behind) where the ring cannot be had.
bool ring_reserve(int64_t slots)
{
    if(ring_slots < slots)
    {
        if(ring != nullptr)
            (void)hipHostFree(ring);
        ring = nullptr;
        ring_slots = 0;
        if(hipHostMalloc((void **)&ring, sizeof(double)*CHUNK*slots,
                    hipHostMallocDefault) != hipSuccess)
        {
            ring = nullptr;
            (void)hipGetLastError();
            return false;
        }
        ring_slots = slots;
    }
    for(int s = 0; s < NSLOT; s++)
        if(ring_ev[s] == nullptr && hipEventCreateWithFlags(&ring_ev[s],
                    hipEventDisableTiming) != hipSuccess)
        {
            ring_ev[s] = nullptr;
            (void)hipGetLastError();
            return false;
        }
    return true;
}

// Copies elements [a, b) of the concatenated arrays to dst; start[q] is the
// place of array q.
void gather(const double *const *src, const std::vector<int64_t> &start,
        int64_t a, int64_t b, double *dst)
{
    size_t q = (size_t)(std::upper_bound(start.begin(), start.end(), a)-
            start.begin())-1;
    while(a < b)
    {
        const int64_t e = std::min(b, start[q+1]);
        if(e > a)
            memcpy(dst, src[q]+(a-start[q]), sizeof(double)*(size_t)(e-a));
        dst += e-a;
        a = e;
        q++;
    }
}

struct Upload
{
    const double *const *src;
    const std::vector<int64_t> &start;
    int64_t total, npieces;
    std::atomic<int64_t> next{0};
    std::mutex mu;
    std::condition_variable cv;
    std::vector<int> left;      // pieces of a chunk not yet packed
    int64_t allowed = ring_slots;   // chunks below this have a free slot
    Upload(const double *const *s, const std::vector<int64_t> &st, int64_t n)
        : src(s), start(st), total(n), npieces((n+PIECE-1)/PIECE)
    {
        const int64_t per = CHUNK/PIECE;
        left.resize((size_t)((n+CHUNK-1)/CHUNK), (int)per);
        left.back() = (int)(npieces-(int64_t)(left.size()-1)*per);
    }
    void work()
    {
        for(;;)
        {
            const int64_t p = next.fetch_add(1);
            if(p >= npieces)
                return;
            const int64_t a = p*PIECE, b = std::min(a+PIECE, total);
            const int64_t c = a/CHUNK;
            {
                std::unique_lock<std::mutex> g(mu);
                cv.wait(g, [&] { return allowed > c; });
            }
            gather(src, start, a, b, ring+(c % ring_slots)*CHUNK+(a-c*CHUNK));
            bool full;
            {
                std::lock_guard<std::mutex> g(mu);
                full = --left[(size_t)c] == 0;
            }
            if(full)
                cv.notify_all();
        }
    }
    void allow(int64_t c)
    {
        {
            std::lock_guard<std::mutex> g(mu);
            allowed = c;
        }
        cv.notify_all();
    }
};

// Returns NO_THREADS, with nothing done, if no thread can be started.
constexpr int NO_THREADS = -100;     // none of the library's codes
int upload_ring(double *d_dst, const double *const *src,
        const std::vector<int64_t> &start, int64_t total)
{
    hipStream_t s = starsh_hip_stream();
    Upload up(src, start, total);
    std::vector<std::thread> threads;
    unsigned nth = std::thread::hardware_concurrency();
    nth = nth < 4 ? 2 : (nth > 16 ? 14 : nth-2);
    // a thread is started for 2 MiB at least
    nth = (unsigned)std::min<int64_t>(nth, std::max<int64_t>(1,
                up.npieces/4));
    // a thread that cannot be started leaves its share to the others
    try
    {
        threads.reserve(nth);
        for(unsigned i = 0; i < nth; i++)
            threads.emplace_back([&up] { up.work(); });
    }
    catch(...)
    {
        if(threads.empty())
            return NO_THREADS;
    }
    hipError_t err = hipSuccess;
    const int64_t nchunks = (int64_t)up.left.size();
    for(int64_t c = 0; c < nchunks && err == hipSuccess; c++)
    {
        {
            std::unique_lock<std::mutex> g(up.mu);
            up.cv.wait(g, [&] { return up.left[(size_t)c] == 0; });
        }
        const int64_t a = c*CHUNK, len = std::min(CHUNK, total-a);
        err = hipMemcpyAsync(d_dst+a, ring+(c % ring_slots)*CHUNK,
                sizeof(double)*(size_t)len, hipMemcpyHostToDevice, s);
        if(err == hipSuccess)
            err = hipEventRecord(ring_ev[c % ring_slots], s);
        // two slots stay on their way while the others are packed
        if(err == hipSuccess && c >= 2)
        {
            err = hipEventSynchronize(ring_ev[(c-2) % ring_slots]);
            up.allow(c-2+ring_slots+1);
        }
    }
    // after an error the copies queued so far still read their slots (and
    // write d_dst, which the caller may free): wait for them before the
    // threads run out and refill the slots
    if(err != hipSuccess)
        (void)hipStreamSynchronize(s);
    up.allow(nchunks);
    for(auto &t : threads)
        t.join();
    HIP_TRY(err);
    HIP_TRY(hipStreamSynchronize(s));
    return STARSH_SUCCESS;
}

} // namespace

// d_dst gets the nseg arrays src[q] of len[q] doubles, one after the other.
extern "C" int hip_upload_segments(double *d_dst, int64_t nseg,
        const double *const *src, const int64_t *len)
{
    try
    {
        std::vector<int64_t> start((size_t)nseg+1, 0);
        for(int64_t q = 0; q < nseg; q++)
            start[(size_t)q+1] = start[(size_t)q]+len[q];
        const int64_t total = start[(size_t)nseg];
        if(total == 0)
            return STARSH_SUCCESS;
        std::unique_lock<std::mutex> g(ring_mu, std::defer_lock);
        if(total > SMALL && g.try_lock())
        {
            if(ring_reserve(std::min<int64_t>(NSLOT, (total+CHUNK-1)/CHUNK)))
            {
                const int info = upload_ring(d_dst, src, start, total);
                if(info != NO_THREADS)
                    return info;
            }
            g.unlock();
        }
        // small, or the ring is in use or cannot be had
        const std::unique_ptr<double[]> h(new double[(size_t)total]);
        gather(src, start, 0, total, h.get());
        return starsh_hip_memcpy_h2d(d_dst, h.get(),
                sizeof(double)*(size_t)total);
    }
    catch(...)
    {
        return STARSH_MALLOC_ERROR;
    }
}

// Frees the ring (no upload may be running).
extern "C" void hip_upload_release(void)
{
    std::lock_guard<std::mutex> g(ring_mu);
    if(ring != nullptr)
        (void)hipHostFree(ring);
    ring = nullptr;
    ring_slots = 0;
}
