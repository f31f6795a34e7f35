// A stand-in for the HIP runtime, for tests of the library's host side without
// a GPU: a program that defines these functions and is linked with the library
// has them called in the runtime's place.  Device memory is host memory, every
// block and stream belongs to a device, kernels are not run (their results
// stay zero), and every piece of work has completed when it is enqueued.  A
// copy, or a free on a stream, of another device's block is counted.
#ifndef FAKE_HIP_HPP
#define FAKE_HIP_HPP

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace fake {
constexpr int kDevices = 2;
struct Block {
    int device;
    size_t bytes;
};
inline std::mutex mu;
inline std::map<char*, Block> blocks;   // device memory, by first byte
inline std::map<void*, int> streams;
inline int foreign = 0;   // uses of a block on another device's stream
inline thread_local int current = 0;

inline void* alloc(size_t bytes, int device)
{
    char* p = (char*)calloc(bytes, 1);
    std::lock_guard<std::mutex> lk(mu);
    blocks[p] = Block{device, bytes};
    return p;
}
inline void release(void* p)
{
    std::lock_guard<std::mutex> lk(mu);
    blocks.erase((char*)p);
    free(p);
}
// the device of the block that holds p, -1 for host memory
inline int device_of(const void* p)
{
    auto it = blocks.upper_bound((char*)p);
    if (it == blocks.begin()) return -1;
    --it;
    return (char*)p < it->first + it->second.bytes ? it->second.device : -1;
}
inline void use(const void* p, void* stream)
{
    std::lock_guard<std::mutex> lk(mu);
    const int d = device_of(p), s = streams.count(stream) ? streams[stream] : -1;
    if (d >= 0 && d != s) {
        foreign++;
        fprintf(stderr, "block of device %d used on a stream of device %d\n", d, s);
    }
}
inline size_t device_bytes(int device)
{
    std::lock_guard<std::mutex> lk(mu);
    size_t s = 0;
    for (auto& b : blocks)
        if (b.second.device == device) s += b.second.bytes;
    return s;
}
} // namespace fake

extern "C" {
int hipGetDeviceCount(int* n) { *n = fake::kDevices; return 0; }
int hipGetDevice(int* d) { *d = fake::current; return 0; }
int hipSetDevice(int d) { fake::current = d; return 0; }
int hipDeviceGetDefaultMemPool(void** pool, int) { *pool = (void*)1; return 0; }
int hipMemPoolSetAttribute(void*, int, void*) { return 0; }
int hipMemPoolTrimTo(void*, size_t) { return 0; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)288 << 30; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned)
{
    *s = malloc(1);
    std::lock_guard<std::mutex> lk(fake::mu);
    fake::streams[*s] = fake::current;
    return 0;
}
int hipStreamDestroy(void* s)
{
    std::lock_guard<std::mutex> lk(fake::mu);
    fake::streams.erase(s);
    free(s);
    return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipEventCreate(void** e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = malloc(1); return 0; }
int hipEventDestroy(void* e) { free(e); return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventQuery(void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0; return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "error"; }
int hipMalloc(void** p, size_t n) { *p = fake::alloc(n, fake::current); return 0; }
int hipFree(void* p) { if (p) fake::release(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(n, 1); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMallocAsync(void** p, size_t n, void* s)
{
    int d;
    {
        std::lock_guard<std::mutex> lk(fake::mu);
        d = fake::streams.count(s) ? fake::streams[s] : fake::current;
    }
    *p = fake::alloc(n, d);
    return 0;
}
int hipFreeAsync(void* p, void* s)
{
    fake::use(p, s);
    fake::release(p);
    return 0;
}
int hipMemcpyAsync(void* dst, const void* src, size_t n, int, void* s)
{
    fake::use(dst, s);
    fake::use(src, s);
    memcpy(dst, src, n);
    return 0;
}
int hipGetSymbolAddress(void** p, const void*) { static char mem[64]; *p = mem; return 0; }
int hipLaunchKernel(const void*, ...) { return 0; }
}

#endif
