// bbx_fetch.h -- particle fields to the host in particle-id order (host side).
#pragma once

#include <algorithm>

#include "bbx_common.h"

namespace bbx {

constexpr int kFetchSlots = 8;                  // chunks in flight
constexpr size_t kFetchRing = 4 * 1024 * 1024;  // bytes; a small solver's ring holds its widest field

struct FetchRing {
    char *ring = nullptr, *d_ring = nullptr;  // pinned, and its device address
    size_t bytes = 0;                         // a flag word follows: the device saw an id outside the set
    char *own = nullptr;                      // the ring's own allocation, after the set has grown
    hipEvent_t ev[kFetchSlots] = {};
};

// A field in storage order: 3 components (vec), 1 or BBX_NFEAT (scal,
// component-major with the solver's stride).
struct FieldSource {
    int width;
    const float4 *vec;
    const float *scal;
};

// run(p, first, count): floats first .. first + count - 1 of the id-ordered
// field; calls for different ranges may come from different threads.
struct FetchTake {
    virtual void run(const float *p, size_t first, size_t count) const = 0;

protected:
    ~FetchTake() = default;
};

// bytes of the ring for a solver of that capacity (and 64 for the flag word)
size_t fetch_ring_bytes(size_t stride);
int fetch_init(bbx_solver *s, char *pinned, char *device, size_t bytes);
void fetch_free(bbx_solver *s);
int fetch_by_id(bbx_solver *s, const FieldSource &f, const FetchTake &take);
// n FP64 vectors (null: zeros) as FP32 rows of dst, the rest of `rows` zero;
// with_ids: row i's fourth word holds i.  Chunk by chunk through the ring: two
// whole host copies cost 7.8 ms in first-touched pages at 1M particles.
int upload_vec4(bbx_solver *s, float4 *dst, const double *xyz, size_t n, size_t rows, bool with_ids);

}  // namespace bbx
