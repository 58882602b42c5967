// nb_download.h -- device-to-host copies of results through pinned pieces.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace nb {

// A callable that outlives the download (held by reference: nothing to allocate).
struct FillRef {
    void *obj;
    int (*call)(void *);
    template <typename F>
    FillRef(F &f) : obj((void *)&f), call([](void *p) { return (*(F *)p)(); }) {}
    int operator()() const { return call(obj); }
};

// A result array on its way to the host: `fill` enqueues the kernel that leaves
// its `count` doubles (caller order) at `src` on the stream.
struct DownField {
    double *dst;          // host; nullptr: not wanted
    const double *src;    // device
    size_t count;
    FillRef fill;
};

// Copies the wanted fields, one after another (they may share src), and returns
// when the last one is in its host array.
int download_fields(const DownField *f, int nf, int dev, hipStream_t s);

// Held by every context and ensemble: the pinned blocks that downloads leave for
// the next one are freed with the last holder.
struct DownloadUse {
    DownloadUse();
    ~DownloadUse();
    DownloadUse(const DownloadUse &) = delete;
    DownloadUse &operator=(const DownloadUse &) = delete;
};

}  // namespace nb
