// The HIP runtime calls of libgpaw_amd.so on the CPU, for tests of its host
// code: memory from malloc, launches and graphs that do nothing, and the n-th
// allocation made to fail.  Loaded with global scope before the library.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <set>

namespace {
std::set<void*> live;
long fail_at = 0, allocations = 0, launches = 0;

int give(void** p, size_t n)
{
    allocations++;
    if (fail_at && allocations == fail_at) return 2;   // hipErrorOutOfMemory
    *p = calloc(1, n ? n : 1);
    live.insert(*p);
    return 0;
}

int take(void* p)
{
    live.erase(p);
    free(p);
    return 0;
}
}  // namespace

extern "C" {
void host_fail_at(long n)   // the n-th allocation from here on; 0: none
{
    fail_at = n;
    allocations = 0;
}
long host_allocations() { return allocations; }
long host_live() { return (long)live.size(); }
long host_launches() { return launches; }

int hipMalloc(void** p, size_t n) { return give(p, n); }
int hipHostMalloc(void** p, size_t n, unsigned) { return give(p, n); }
int hipFree(void* p) { return take(p); }
int hipHostFree(void* p) { return take(p); }
int hipMallocAsync(void** p, size_t n, void*) { return give(p, n); }
int hipFreeAsync(void* p, void*) { return take(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipLaunchKernel(const void*, uint64_t, uint32_t, uint64_t, uint32_t, void**, size_t, void*)
{
    launches++;
    return 0;
}
int hipEventCreate(void** e) { return give(e, 1); }
int hipEventCreateWithFlags(void** e, unsigned) { return give(e, 1); }
int hipEventDestroy(void* e) { return take(e); }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipGraphCreate(void** g, unsigned) { return give(g, 1); }
int hipGraphDestroy(void* g) { return take(g); }
int hipGraphAddKernelNode(void** n, void*, const void**, size_t, const void*)
{
    *n = n;
    return 0;
}
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { return give(e, 1); }
int hipGraphExecDestroy(void* e) { return take(e); }
int hipGraphLaunch(void*, void*) { return 0; }
}
