// Staged transfers between rows of device memory and a padded host array.
//
// The host arrays are pageable and padded, so a direct copy either runs row by
// row or goes through a temporary of the whole state (whose pages are touched
// for the first time at every call).  Here chunks of whole rows go through
// pinned buffers kept by their owner: while one chunk is on the link, the rows
// of another are moved between its buffer and the host array.  Large states
// are moved by several threads, each with two buffers, because one thread
// moves host memory several times slower than the link delivers it.  Small
// states take buffers of a sixteenth of their size (pinning memory costs about
// 0.4 ms per MB, paid once per owner).  Measured, 40 steps of a 256^3 solver and
// the return of its 671 MB state: 1024 ms through a temporary, 840 ms so.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>

#include "cles_internal.h"

namespace cles {

namespace {
constexpr size_t STAGE_CHUNK = (size_t)4 << 20;    // bytes per buffer at most
constexpr size_t STAGE_SMALL = (size_t)256 << 10;  // ... and at least
constexpr size_t STAGE_LANE = (size_t)16 << 20;    // bytes of state per thread
constexpr int STAGE_LANES = 6;                     // threads at most

void check(hipError_t e, const char *what)
{
    if (e != hipSuccess) throw Error{CLES_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e)};
}
}  // namespace

DeviceScope::DeviceScope(int device)
{
    int now = -1;
    check(hipGetDevice(&now), "hipGetDevice");
    if (now == device) return;
    check(hipSetDevice(device), "hipSetDevice");
    before = now;
}

DeviceScope::~DeviceScope()
{
    if (before >= 0) (void)hipSetDevice(before);
}

PinnedBuf::~PinnedBuf() { release(); }

void PinnedBuf::release()
{
    if (ptr) {
        if (pinned) (void)hipHostFree(ptr);
        else std::free(ptr);
    }
    ptr = nullptr;
    cap = 0;
}

void *PinnedBuf::get(size_t bytes)
{
    if (cap >= bytes) return ptr;
    release();
    if (hipHostMalloc(&ptr, bytes, hipHostMallocDefault) == hipSuccess) {
        pinned = true;
    } else {   // no pinned memory left: pageable works with the same copies
        (void)hipGetLastError();
        ptr = std::malloc(bytes);
        pinned = false;
        if (!ptr) throw std::bad_alloc();
    }
    cap = bytes;
    return ptr;
}

HostStage::~HostStage()
{
    for (auto &l : lanes)
        for (hipEvent_t e : l->ev)
            if (e) (void)hipEventDestroy(e);
}

void HostStage::transfer(bool down, int device, hipStream_t st, double *dev, const View3 &host_view, int64_t ncomp,
                         int64_t comp_stride, double *host)
{
    std::lock_guard<std::mutex> lk(mu);
    const int64_t n0 = host_view.n[0], n1 = host_view.n[1], n2 = host_view.n[2];
    const int64_t nrows = ncomp * n1 * n2;
    const size_t row = (size_t)n0 * sizeof(double), total = row * (size_t)nrows;
    const size_t chunk = std::min(STAGE_CHUNK, std::max(STAGE_SMALL, total / 16));
    const int64_t per = std::max<int64_t>(1, (int64_t)(chunk / row));   // rows per chunk
    const int64_t nchunk = (nrows + per - 1) / per;
    const int nlane = (int)std::min<int64_t>(std::min<int64_t>(STAGE_LANES, 1 + (int64_t)(total / STAGE_LANE)), nchunk);
    while ((int)lanes.size() < nlane) lanes.emplace_back(new Lane);
    auto host_row = [&](int64_t r) -> double * {
        const int64_t c = r / (n1 * n2), q = r - c * n1 * n2, k = q / n1, j = q - k * n1;
        return host + c * comp_stride + j * host_view.s[1] + k * host_view.s[2];
    };
    auto work = [&](int w) {
        Lane &l = *lanes[w];
        for (int b = 0; b < 2; b++)
            if (!l.ev[b]) check(hipEventCreateWithFlags(&l.ev[b], hipEventDisableTiming), "hipEventCreate");
        auto first = [&](int64_t i) { return (w + i * nlane) * per; };
        auto rows = [&](int64_t i) { return std::min<int64_t>(per, nrows - first(i)); };
        const int64_t mine = (nchunk - w + nlane - 1) / nlane;
        // both buffers in one allocation (each costs about 0.1 ms to pin)
        const size_t half = row * (size_t)std::min<int64_t>(per, nrows);
        char *const base = (char *)l.buf.get(half * (size_t)std::min<int64_t>(2, mine));
        auto buf = [&](int64_t i) { return base + half * (size_t)(i & 1); };
        auto issue = [&](int64_t i) {
            char *b = buf(i);
            double *d = dev + first(i) * n0;
            const size_t bytes = row * (size_t)rows(i);
            if (down) check(hipMemcpyAsync(b, d, bytes, hipMemcpyDeviceToHost, st), "hipMemcpyAsync");
            else check(hipMemcpyAsync(d, b, bytes, hipMemcpyHostToDevice, st), "hipMemcpyAsync");
            check(hipEventRecord(l.ev[i & 1], st), "hipEventRecord");
        };
        auto move = [&](int64_t i) {
            char *b = buf(i);
            for (int64_t r = 0; r < rows(i); r++) {
                double *h = host_row(first(i) + r);
                if (down) std::memcpy(h, b + row * (size_t)r, row);
                else std::memcpy(b + row * (size_t)r, h, row);
            }
        };
        if (down)
            for (int64_t i = 0; i < std::min<int64_t>(2, mine); i++) issue(i);
        for (int64_t i = 0; i < mine; i++) {
            if (down) {
                check(hipEventSynchronize(l.ev[i & 1]), "hipEventSynchronize");
                move(i);
                if (i + 2 < mine) issue(i + 2);
            } else {
                if (i >= 2) check(hipEventSynchronize(l.ev[i & 1]), "hipEventSynchronize");
                move(i);
                issue(i);
            }
        }
    };
    std::vector<std::thread> pool;
    std::vector<Error> failed((size_t)nlane, Error{CLES_OK, ""});
    auto guarded = [&](int w) {
        try {
            DeviceScope on(device);   // lane 0 and lanes without a thread run on the caller's
            work(w);
        } catch (const Error &e) {
            failed[w] = e;
        } catch (const std::exception &) {
            failed[w] = Error{CLES_ERR_NOMEM, "host allocation failed"};
        }
    };
    int started = 1;
    try {
        for (; started < nlane; started++) pool.emplace_back(guarded, started);
    } catch (const std::exception &) {   // no more threads: this one does their share
    }
    guarded(0);
    for (int w = started; w < nlane; w++) guarded(w);
    for (auto &t : pool) t.join();
    const hipError_t e = hipStreamSynchronize(st);
    for (const Error &f : failed)
        if (f.code != CLES_OK) throw f;
    check(e, "hipStreamSynchronize");
}

}  // namespace cles
