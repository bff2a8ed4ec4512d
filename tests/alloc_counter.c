/* Counts the calls of the HIP runtime's allocators that libmmsim makes: loaded with global symbols before the library,
 * its definitions are the ones the library's calls find; they pass the calls on.  Only tests load it. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static long counted;
long allocator_calls(void) { return counted; }

static void *runtime(const char *name) {
    static void *lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    return lib ? dlsym(lib, name) : NULL;
}
#define PASS_ON(name, params, ...)                 \
    int name params {                              \
        int(*next) params = runtime(#name);        \
        ++counted;                                 \
        return next ? next(__VA_ARGS__) : 1;       \
    }
PASS_ON(hipMalloc, (void **p, size_t n), p, n)
PASS_ON(hipFree, (void *p), p)
PASS_ON(hipHostMalloc, (void **p, size_t n, unsigned flags), p, n, flags)
PASS_ON(hipHostFree, (void *p), p)
