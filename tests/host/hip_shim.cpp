// Runtime calls that fail on request or are counted, for tests of error paths
// and fallbacks: loaded with RTLD_GLOBAL before liblbm.so, its definitions are
// the ones liblbm.so binds to.  Nothing here reaches the GPU by itself.
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>

#include <new>

extern "C" {

int shim_fail_host_malloc = 0;      // hipHostMalloc: out of memory
int shim_host_mallocs = 0;           // hipHostMalloc calls for 4 MiB and more so far
int shim_launches = 0;               // kernels launched so far
int shim_copies = 0;                 // hipMemcpyAsync calls so far
int shim_streams = 0;                // streams created so far
int shim_last_gone = 0;              // number, in the order of creation, of the stream destroyed last
int shim_fail_query = 0;             // hipStreamQuery: so many calls fail ...
int shim_fail_query_from = 0;        // ... once so many kernels have been launched
unsigned long long shim_fail_new = 0; // operator new of exactly so many bytes throws
unsigned long long shim_malloc_bytes = 0; // bytes asked of hipMalloc so far

static void *streams[64]; // the latest ones, by number

static void *real(const char *name)
{
    static void *lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    return lib ? dlsym(lib, name) : nullptr;
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    if (shim_fail_host_malloc)
        return 2; // hipErrorOutOfMemory
    if (bytes >= 4u << 20)
        shim_host_mallocs++;
    static auto f = (int (*)(void **, size_t, unsigned))real("hipHostMalloc");
    return f(p, bytes, flags);
}

int hipStreamQuery(void *stream)
{
    if (shim_fail_query > 0 && shim_launches >= shim_fail_query_from) {
        shim_fail_query--;
        return 999; // hipErrorUnknown
    }
    static auto f = (int (*)(void *))real("hipStreamQuery");
    return f(stream);
}

int hipMalloc(void **p, size_t bytes)
{
    shim_malloc_bytes += bytes;
    static auto f = (int (*)(void **, size_t))real("hipMalloc");
    return f(p, bytes);
}

int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *stream)
{
    shim_copies++;
    static auto f = (int (*)(void *, const void *, size_t, int, void *))real("hipMemcpyAsync");
    return f(dst, src, bytes, kind, stream);
}

int hipStreamCreateWithFlags(void **stream, unsigned flags)
{
    static auto f = (int (*)(void **, unsigned))real("hipStreamCreateWithFlags");
    const int rc = f(stream, flags);
    if (rc == 0)
        streams[shim_streams++ % 64] = *stream;
    return rc;
}

int hipStreamDestroy(void *stream)
{
    for (int k = shim_streams - 1; k >= 0 && k > shim_streams - 64; k--)
        if (streams[k % 64] == stream) {
            shim_last_gone = k;
            break;
        }
    static auto f = (int (*)(void *))real("hipStreamDestroy");
    return f(stream);
}

struct Dim3 {
    unsigned x, y, z;
};

int hipLaunchKernel(const void *kernel, Dim3 grid, Dim3 block, void **args, size_t lds, void *stream)
{
    shim_launches++;
    static auto f = (int (*)(const void *, Dim3, Dim3, void **, size_t, void *))real("hipLaunchKernel");
    return f(kernel, grid, block, args, lds, stream);
}

} // extern "C"

void *operator new(size_t bytes)
{
    void *p = shim_fail_new && bytes == shim_fail_new ? nullptr : malloc(bytes ? bytes : 1);
    if (!p)
        throw std::bad_alloc();
    return p;
}

void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
