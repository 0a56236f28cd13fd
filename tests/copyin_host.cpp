// Host driver of the factor upload (csrc/hip/copyin.hip, compiled for the
// host alone) with the runtime calls it makes replaced by the ones below: a
// "device" in host memory, copies that are carried out when they are waited
// for, and failures on request.  Argument: ok, pin (no pinned memory), thread
// (no thread can be started) or copy (the fourth copy fails).  Prints the
// returned value, whether the data arrived, the copies still queued on return
// and the slots that changed while a copy from them was queued.
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <dlfcn.h>
#include <errno.h>
#include <deque>
#include <vector>

extern "C" int hip_upload_segments(double *, int64_t, const double *const *,
        const int64_t *);

namespace {

struct Copy
{
    void *dst;
    const void *src;
    size_t bytes;
    unsigned long long sum;
    int id;
};
std::deque<Copy> queue;
int mode_pin, mode_thread, mode_copy, copies, changed, last_id;
int event_id[64], events;

// A checksum of a few words of every page.
unsigned long long sum_of(const void *p, size_t bytes)
{
    const unsigned long long *w = (const unsigned long long *)p;
    unsigned long long s = 0;
    for(size_t i = 0; i < bytes/8; i += 257)
        s = s*31+w[i];
    return s;
}

void drain(int upto)
{
    while(!queue.empty() && queue.front().id <= upto)
    {
        const Copy c = queue.front();
        queue.pop_front();
        changed += sum_of(c.src, c.bytes) != c.sum;
        memcpy(c.dst, c.src, c.bytes);
    }
}

} // namespace

extern "C" {

hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    if(mode_pin)
        return hipErrorOutOfMemory;
    *p = malloc(bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t)(event_id+events++);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    *(int *)e = last_id;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    drain(*(int *)e);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    drain(last_id);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes,
        hipMemcpyKind, hipStream_t)
{
    if(mode_copy && ++copies == 4)
        return hipErrorUnknown;
    queue.push_back(Copy{dst, src, bytes, sum_of(src, bytes), ++last_id});
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused by the test"; }
hipStream_t starsh_hip_stream(void) { return nullptr; }
int starsh_hip_memcpy_h2d(void *dst, const void *src, size_t bytes)
{
    drain(last_id);
    memcpy(dst, src, bytes);
    return 0;
}

int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *),
        void *x)
{
    using fn = int (*)(pthread_t *, const pthread_attr_t *,
            void *(*)(void *), void *);
    if(mode_thread)
        return EAGAIN;
    return ((fn)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, x);
}

}

int main(int, char **argv)
{
    mode_pin = !strcmp(argv[1], "pin");
    mode_thread = !strcmp(argv[1], "thread");
    mode_copy = !strcmp(argv[1], "copy");
    // 11 slots' worth (the ring has 8), in arrays of odd lengths
    const int64_t slot = (int64_t)1 << 21, total = 11*slot+5, n = 7;
    std::vector<double> data((size_t)total), dev((size_t)total);
    for(int64_t i = 0; i < total; i++)
        data[(size_t)i] = (double)i;
    const double *src[7];
    int64_t len[7], at = 0;
    for(int64_t q = 0; q < n; q++)
    {
        len[q] = q+1 < n ? total/n-q*1001 : total-at;
        src[q] = data.data()+at;
        at += len[q];
    }
    const int info = hip_upload_segments(dev.data(), n, src, len);
    const int left = (int)queue.size();
    drain(last_id);
    printf("%d %d %d %d\n", info, (int)(dev == data), left, changed);
    return 0;
}
