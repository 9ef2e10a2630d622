/* Stands before the HIP runtime in a test's process and forces what a test
 * cannot bring about through the library: allocations that fail, a byte that
 * changes on its way to the device.  Loaded with RTLD_GLOBAL before the
 * library, so that the library's calls come here first. */
#include <dlfcn.h>
#include <stddef.h>
#include <string.h>

typedef int (*malloc_fn)(void **, size_t);
typedef int (*free_fn)(void *);
typedef int (*host_malloc_fn)(void **, size_t, unsigned);
typedef int (*copy_fn)(void *, const void *, size_t, int, void *);

static void *hip;
int faults_host_malloc;                          /* > 0: the next ones fail */
size_t faults_copy_bytes, faults_copy_offset;    /* the next async upload of that many bytes ... */
int faults_copy_word;                            /* ... holds this word at that offset */

void faults_init(const char *runtime) { hip = dlopen(runtime, RTLD_NOW | RTLD_NOLOAD); }
static void *real(const char *name) { return dlsym(hip, name); }

size_t faults_live, faults_peak;     /* device bytes allocated through here */
size_t faults_budget, faults_refuse; /* if set: no more live bytes than this; no allocation of this size */
static struct {
    void *p;
    size_t bytes;
} block[4096];

int hipMalloc(void **p, size_t bytes) {
    *p = NULL;
    if ((faults_budget && faults_live + bytes > faults_budget) || (faults_refuse && bytes == faults_refuse))
        return 2; /* hipErrorOutOfMemory */
    const int e = ((malloc_fn)real("hipMalloc"))(p, bytes);
    for (int k = 0; !e && k < 4096; k++)
        if (!block[k].p) {
            block[k].p = *p;
            block[k].bytes = bytes;
            faults_live += bytes;
            if (faults_live > faults_peak) faults_peak = faults_live;
            break;
        }
    return e;
}

int hipFree(void *p) {
    for (int k = 0; p && k < 4096; k++)
        if (block[k].p == p) {
            block[k].p = NULL;
            faults_live -= block[k].bytes;
        }
    return ((free_fn)real("hipFree"))(p);
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    if (faults_host_malloc > 0) {
        faults_host_malloc--;
        *p = NULL;
        return 2; /* hipErrorOutOfMemory */
    }
    return ((host_malloc_fn)real("hipHostMalloc"))(p, bytes, flags);
}

int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *stream) {
    if (kind == 1 && faults_copy_bytes && bytes == faults_copy_bytes) {
        memcpy((char *)src + faults_copy_offset, &faults_copy_word, sizeof(int));
        faults_copy_bytes = 0;
    }
    return ((copy_fn)real("hipMemcpyAsync"))(dst, src, bytes, kind, stream);
}
