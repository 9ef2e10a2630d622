/* Stands before the HIP runtime in a test's process and forces what a test
 * cannot bring about through the library: allocations that fail, a byte that
 * changes on its way to the device.  Loaded with RTLD_GLOBAL before the
 * library, so that the library's calls come here first. */
#include <dlfcn.h>
#include <stddef.h>
#include <string.h>

typedef int (*host_malloc_fn)(void **, size_t, unsigned);
typedef int (*copy_fn)(void *, const void *, size_t, int, void *);

static void *hip;
int faults_host_malloc;                          /* > 0: the next ones fail */
size_t faults_copy_bytes, faults_copy_offset;    /* the next async upload of that many bytes ... */
int faults_copy_word;                            /* ... holds this word at that offset */

void faults_init(const char *runtime) { hip = dlopen(runtime, RTLD_NOW | RTLD_NOLOAD); }
static void *real(const char *name) { return dlsym(hip, name); }

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
