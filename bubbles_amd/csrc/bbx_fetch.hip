// bbx_fetch.hip -- particle fields to the host in particle-id order, and a
// new solver's particles to the device.
//
// A field lies in storage (cell) order.  Sorting it out on the host took a
// download of the id table, one of the field, and a scatter through both:
// 65 us for 2k vectors, 104 us for 16k, 5.1 ms for 1M and 34 ms for 3.2M,
// whose scatter leaves the host's caches.  Here the device puts the field in
// id order as packed FP32 and the host only widens it.  A field that fits
// the pinned ring goes there straight from the kernel (262k vectors in
// 39 us; a device buffer and a copy of it took 77); a larger one goes to the
// half of the position ping-pong that holds nothing between calls, and comes
// in chunks while the host widens those before.
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "bbx_fetch.h"

namespace bbx {

// dst[(id - lo) * W + w] = component w of particle id, for ids in [lo, hi).
// Neighbouring slots hold mostly neighbouring ids, so the scattered stores
// meet in the same cache lines.
template <int W>
__global__ void __launch_bounds__(kBlock) k_by_id(const float4 *__restrict__ pos, const float4 *__restrict__ vec,
                                                  const float *__restrict__ scal, int stride, int n, int lo, int hi,
                                                  float *__restrict__ dst, int *bad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int id = __float_as_int(pos[i].w);
    if (id < 0 || id >= n) {
        __hip_atomic_store(bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    if (id < lo || id >= hi) return;
    float *d = dst + (size_t)(id - lo) * W;
    if constexpr (W == 3) {
        const float4 v = vec[i];
        d[0] = v.x;
        d[1] = v.y;
        d[2] = v.z;
    } else if constexpr (W == 1) {
        d[0] = scal[i];
    } else {
        float4 *d4 = reinterpret_cast<float4 *>(d);
        for (int f = 0; f < W; f += 4)
            d4[f / 4] = make_float4(scal[(size_t)f * stride + i], scal[(size_t)(f + 1) * stride + i],
                                    scal[(size_t)(f + 2) * stride + i], scal[(size_t)(f + 3) * stride + i]);
    }
}

static int launch_by_id(bbx_solver *s, const FieldSource &f, int lo, int hi, float *dst) {
    const unsigned nb = (unsigned)((s->n + kBlock - 1) / kBlock);
    int *bad = (int *)(s->fetch->d_ring + s->fetch->bytes);
    if (f.width == 3)
        k_by_id<3><<<nb, kBlock, 0, s->stream>>>(s->posA, f.vec, nullptr, s->stride, s->n, lo, hi, dst, bad);
    else if (f.width == 1)
        k_by_id<1><<<nb, kBlock, 0, s->stream>>>(s->posA, nullptr, f.scal, s->stride, s->n, lo, hi, dst, bad);
    else
        k_by_id<BBX_NFEAT><<<nb, kBlock, 0, s->stream>>>(s->posA, nullptr, f.scal, s->stride, s->n, lo, hi, dst, bad);
    BBX_HIP_CHECK(hipGetLastError());
    return BBX_OK;
}

size_t fetch_ring_bytes(size_t stride) {
    const size_t want = (stride * BBX_NFEAT * sizeof(float) + 4095) / 4096 * 4096;
    return want < kFetchRing ? want : kFetchRing;
}

int fetch_init(bbx_solver *s, char *pinned, char *device, size_t bytes) {
    if (!s->fetch) s->fetch = new FetchRing();
    FetchRing *r = s->fetch;
    r->ring = pinned;
    r->d_ring = device;
    r->bytes = bytes;
    for (int k = 0; k < kFetchSlots; k++)
        if (!r->ev[k] && hipEventCreateWithFlags(&r->ev[k], hipEventDisableTiming) != hipSuccess)
            return fail(BBX_E_HIP, "event create");
    return BBX_OK;
}

void fetch_free(bbx_solver *s) {
    FetchRing *r = s->fetch;
    if (!r) return;
    for (hipEvent_t e : r->ev)
        if (e) (void)hipEventDestroy(e);
    if (r->own) (void)hipHostFree(r->own);
    delete r;
    s->fetch = nullptr;
}

// A larger ring for a set that has grown; without one the smaller one serves.
// Not before a field wants it: pinned memory of 2 MB or more takes 300 us.
static void fetch_grow(bbx_solver *s) {
    FetchRing *r = s->fetch;
    const size_t want = fetch_ring_bytes((size_t)s->stride);
    if (r->bytes >= want) return;
    char *p = nullptr, *d = nullptr;
    if (hipHostMalloc((void **)&p, want + 64, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess ||
        hipHostGetDevicePointer((void **)&d, p, 0) != hipSuccess) {
        if (p) (void)hipHostFree(p);
        (void)hipGetLastError();
        return;
    }
    if (r->own) (void)hipHostFree(r->own);
    r->own = r->ring = p;
    r->d_ring = d;
    r->bytes = want;
}

// what the kernel saw of the id table; the field is not given out where it is corrupt
static int check_ids(const bbx_solver *s) {
    const FetchRing *r = s->fetch;
    if (__atomic_load_n((const int *)(r->ring + r->bytes), __ATOMIC_ACQUIRE))
        return fail(BBX_E_INVALID, "corrupt particle id table");
    return BBX_OK;
}

namespace {

// Below this many floats the threads' start costs more than they save: with
// four helpers 0.8M floats take 0.26 ms either way, 3.1M 0.74 ms instead of
// 1.30, 9.6M 2.4 ms instead of 5.2; eight helpers gain little more.
constexpr size_t kFetchHelpersFrom = 1500000;
constexpr int kFetchHelpers = 4;

// Copy `total` floats at `src` (device) through the ring; take(p, first,
// count) gets them in host memory, in chunks, each once.  With helpers the
// chunks of a large field are taken by several threads at a time.
struct Pipe {
    bbx_solver *s;
    const float *src;
    size_t total, per;  // floats, floats per chunk
    int chunks;
    const FetchTake *take;
    size_t base;        // float index of src[0] in the field

    size_t count(int c) const { return std::min(per, total - (size_t)c * per); }
    float *slot(int c) const { return (float *)(s->fetch->ring + (size_t)(c % kFetchSlots) * (s->fetch->bytes / kFetchSlots)); }
    void consume(int c) const { take->run(slot(c), base + (size_t)c * per, count(c)); }
    int send(int c) const {
        BBX_HIP_CHECK(hipMemcpyAsync(slot(c), src + (size_t)c * per, sizeof(float) * count(c), hipMemcpyDeviceToHost, s->stream));
        BBX_HIP_CHECK(hipEventRecord(s->fetch->ev[c % kFetchSlots], s->stream));
        return BBX_OK;
    }
    // before any chunk is taken: the kernel has looked at every id by then
    int arrive(int c) const {
        BBX_HIP_CHECK(hipEventSynchronize(s->fetch->ev[c % kFetchSlots]));
        return check_ids(s);
    }
    int one_thread() const {
        for (int c = 0; c < std::min(chunks, kFetchSlots); c++) BBX_CHECK(send(c));
        for (int c = 0; c < chunks; c++) {
            BBX_CHECK(arrive(c));
            consume(c);
            if (c + kFetchSlots < chunks) BBX_CHECK(send(c + kFetchSlots));
        }
        return BBX_OK;
    }
    // This thread sends and waits, helper h takes chunks h, h + kFetchHelpers, ...
    // A slot is refilled once its chunk has been taken.
    int with_helpers() const {
        std::atomic<int> ready{0};              // chunks that have arrived
        std::atomic<int> taken[kFetchSlots];    // per slot: its last taken chunk + 1
        for (auto &t : taken) t.store(0, std::memory_order_relaxed);
        std::atomic<bool> stop{false};
        std::thread th[kFetchHelpers];
        auto take_chunk = [&](int c) {
            consume(c);
            taken[c % kFetchSlots].store(c + 1, std::memory_order_release);
        };
        auto work = [&](int h) {
            for (int c = h; c < chunks; c += kFetchHelpers) {
                while (ready.load(std::memory_order_acquire) <= c) {
                    if (stop.load(std::memory_order_relaxed)) return;
                    std::this_thread::yield();
                }
                take_chunk(c);
            }
        };
        int started = 0;
        try {
            for (; started < kFetchHelpers; started++) th[started] = std::thread(work, started);
        } catch (const std::exception &) {  // no more threads: this one takes their chunks
        }
        auto feed = [&]() -> int {
            for (int c = 0; c < std::min(chunks, kFetchSlots); c++) BBX_CHECK(send(c));
            for (int c = 0; c < chunks; c++) {
                BBX_CHECK(arrive(c));
                ready.store(c + 1, std::memory_order_release);
                if (c % kFetchHelpers >= started) take_chunk(c);
                if (c + kFetchSlots < chunks) {
                    while (taken[c % kFetchSlots].load(std::memory_order_acquire) != c + 1) std::this_thread::yield();
                    BBX_CHECK(send(c + kFetchSlots));
                }
            }
            return BBX_OK;
        };
        const int rc = feed();
        if (rc != BBX_OK) stop.store(true);
        for (int h = 0; h < started; h++) th[h].join();
        return rc;
    }
};

}  // namespace

int fetch_by_id(bbx_solver *s, const FieldSource &f, const FetchTake &take) {
    if (s->n == 0) return BBX_OK;
    FetchRing *r = s->fetch;
    const size_t all = (size_t)s->n * f.width;
    if (all * sizeof(float) > r->bytes) fetch_grow(s);
    __atomic_store_n((int *)(r->ring + r->bytes), 0, __ATOMIC_RELEASE);
    if (all * sizeof(float) <= r->bytes) {
        BBX_CHECK(launch_by_id(s, f, 0, s->n, (float *)r->d_ring));
        BBX_HIP_CHECK(hipStreamSynchronize(s->stream));
        BBX_CHECK(check_ids(s));
        take.run((const float *)r->ring, 0, all);
    } else {
        // posB holds nothing between calls: 4 floats a particle
        float *scratch = reinterpret_cast<float *>(s->posB);
        const int ids = (int)std::min<size_t>((size_t)s->n, (size_t)s->stride * 4 / (size_t)f.width);
        for (int lo = 0; lo < s->n; lo += ids) {
            const int hi = std::min(s->n, lo + ids);
            BBX_CHECK(launch_by_id(s, f, lo, hi, scratch));
            Pipe p{s, scratch, (size_t)(hi - lo) * f.width, r->bytes / kFetchSlots / sizeof(float), 0, &take, (size_t)lo * f.width};
            p.chunks = (int)((p.total + p.per - 1) / p.per);
            const int rc = p.total >= kFetchHelpersFrom ? p.with_helpers() : p.one_thread();
            if (rc != BBX_OK) {
                (void)hipStreamSynchronize(s->stream);  // no copy into the ring is left behind
                return rc;
            }
        }
    }
    return BBX_OK;
}

int upload_vec4(bbx_solver *s, float4 *dst, const double *xyz, size_t n, size_t rows, bool with_ids) {
    FetchRing *r = s->fetch;
    const size_t slot = r->bytes / kFetchSlots, per = slot / sizeof(float4);
    size_t c = 0;
    for (size_t lo = 0; lo < rows; lo += per, c++) {
        const int k = (int)(c % kFetchSlots);
        if (c >= (size_t)kFetchSlots) BBX_HIP_CHECK(hipEventSynchronize(r->ev[k]));  // its last chunk has gone
        float4 *h = (float4 *)(r->ring + (size_t)k * slot);
        const size_t hi = std::min(rows, lo + per);
        for (size_t i = lo; i < hi; i++) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < n && xyz) v = make_float4((float)xyz[3 * i], (float)xyz[3 * i + 1], (float)xyz[3 * i + 2], 0.f);
            if (i < n && with_ids) {
                const int id = (int)i;
                std::memcpy(&v.w, &id, sizeof(int));
            }
            h[i - lo] = v;
        }
        BBX_HIP_CHECK(hipMemcpyAsync(dst + lo, h, sizeof(float4) * (hi - lo), hipMemcpyHostToDevice, s->stream));
        BBX_HIP_CHECK(hipEventRecord(r->ev[k], s->stream));
    }
    BBX_HIP_CHECK(hipStreamSynchronize(s->stream));
    return BBX_OK;
}

}  // namespace bbx
