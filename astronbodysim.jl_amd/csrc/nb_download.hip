// nb_download.hip -- device-to-host copies of results through pinned pieces.
//
// A copy into a program's own (pageable) array is a staged copy with one
// synchronisation per array, 30 to 40 us however small, and on large arrays one
// host thread that moves the bytes and takes the page faults of a new array at
// about 10 GB/s.  Here the arrays go through DL_SLOTS pinned pieces of DL_PIECE
// bytes: a kernel writes a piece over PCIe (27 us less than a copy command for
// two small arrays) while the host empties those before it, and results of
// DL_SLOTS pieces or more are emptied by several threads, which is where the
// page faults of a new array cost most (two arrays of 3.6 MB, eight pieces: by
// one thread 1.49 ms into new memory and 0.29 into used, by four 0.88 and 0.25;
// six pieces 0.22 and 0.23).
// Positions and velocities into new arrays, before -> after: 1000 particles
// 69 -> 29 us, 4096 130 -> 33, 16001 82 -> 50, 65536 213 -> 135, 2^20
// 5.2 -> 1.8 ms, 2.1e6 10.3 -> 3.5 ms (one thread 8.7, two 5.2, eight 3.4).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <new>
#include <thread>

#include "nb_download.h"
#include "nb_idle_pool.h"
#include "nb_internal.h"

namespace nb {

namespace {

constexpr size_t DL_PIECE = (size_t)1 << 20;
constexpr int DL_SLOTS = 8;
constexpr int DL_THREADS = 4;

struct Block {
    int dev = 0;
    char *mem = nullptr;
    hipEvent_t ev[DL_SLOTS] = {};
    Block *next = nullptr;
};

// Idle blocks while any context or ensemble lives.
IdlePool<Block, 4> g_pool;

void free_block(Block *b) {
    if (!b) return;
    for (hipEvent_t e : b->ev)
        if (e) (void)hipEventDestroy(e);
    if (b->mem) (void)hipHostFree(b->mem);
    delete b;
}

// nullptr when the host has no pinned memory left.
Block *take_block(int dev) {
    if (Block *idle = g_pool.take(dev)) return idle;
    Block *b = new (std::nothrow) Block;
    if (!b) return nullptr;
    b->dev = dev;
    bool ok = hipHostMalloc((void **)&b->mem, DL_PIECE * DL_SLOTS,
                            hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess;
    if (!ok) b->mem = nullptr;
    for (int k = 0; k < DL_SLOTS && ok; ++k)
        ok = hipEventCreateWithFlags(&b->ev[k], hipEventDisableTiming | hipEventReleaseToSystem) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        free_block(b);
        return nullptr;
    }
    return b;
}

// Coalesced stores to pinned host memory: one launch instead of a copy command.
__global__ __launch_bounds__(256) void k_to_pinned(const double *__restrict__ src, double *__restrict__ dst,
                                                   size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

struct Piece {
    int field;
    size_t at, count;   // doubles
};

// The pieces of the fields in the mask `todo`, in order.
struct Pieces {
    const DownField *f;
    int nf;
    unsigned todo;
    int field = -1;
    size_t at = 0;
    bool next(Piece &p) {
        while (field < 0 || at >= f[field].count) {
            do {
                if (++field >= nf) return false;
            } while (!(todo >> field & 1));
            at = 0;
        }
        p.field = field;
        p.at = at;
        p.count = std::min(f[field].count - at, DL_PIECE / sizeof(double));
        at += p.count;
        return true;
    }
};

int copy_direct(const DownField &f, hipStream_t s) {
    NB_TRY(f.fill());
    NB_HIP(hipMemcpyAsync(f.dst, f.src, sizeof(double) * f.count, hipMemcpyDeviceToHost, s));
    NB_HIP(hipStreamSynchronize(s));
    return NB_OK;
}

// Whether p is memory of the HIP runtime's own (pinned, managed, device).
bool runtime_memory(const void *p) {
    hipPointerAttribute_t at{};
    const hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess && at.type != hipMemoryTypeUnregistered;
}

int copy_pieces(const DownField *f, int nf, unsigned todo, Block *b, size_t npieces, hipStream_t s) {
    // Worker t empties the pieces t, t + DL_THREADS, ... once `ready` has passed
    // them.  The workers start with the first piece's arrival, not before: they
    // wait in a loop, and the device may still have a whole run ahead of it.
    std::atomic<size_t> ready{0};
    std::atomic<size_t> emptied[DL_SLOTS];   // pieces emptied from each slot
    for (auto &e : emptied) e.store(0, std::memory_order_relaxed);
    std::atomic<bool> stop{false};
    auto empty = [&](const Piece &p, size_t k) {
        memcpy(f[p.field].dst + p.at, b->mem + (k % DL_SLOTS) * DL_PIECE, p.count * sizeof(double));
        emptied[k % DL_SLOTS].fetch_add(1, std::memory_order_release);
    };
    auto worker = [&](int t) {
        Pieces it{f, nf, todo};
        Piece p;
        for (size_t k = 0; it.next(p); ++k) {
            if ((int)(k % DL_THREADS) != t) continue;
            while (ready.load(std::memory_order_acquire) <= k) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            empty(p, k);
        }
    };
    std::thread threads[DL_THREADS];
    int started = 0;   // (none: the calling thread empties the pieces)
    auto start_workers = [&] {
        try {
            for (; started < DL_THREADS; ++started) threads[started] = std::thread(worker, started);
        } catch (...) {   // no thread or no memory for one
            stop.store(true);
            for (int t = 0; t < started; ++t) threads[t].join();
            started = 0;
            stop.store(false);
        }
    };
    int rc = NB_OK;
    Pieces sent{f, nf, todo}, got{f, nf, todo};
    Piece p;
    size_t nsent = 0;
    auto send = [&]() -> int {
        if (!sent.next(p)) return NB_OK;
        const size_t slot = nsent % DL_SLOTS;
        if (p.at == 0) NB_TRY(f[p.field].fill());
        double *to = (double *)(b->mem + slot * DL_PIECE);
        k_to_pinned<<<(unsigned)std::min<size_t>((p.count + 255) / 256, 256), 256, 0, s>>>(f[p.field].src + p.at, to,
                                                                                          p.count);
        NB_HIP(hipGetLastError());
        NB_HIP(hipEventRecord(b->ev[slot], s));
        ++nsent;
        return NB_OK;
    };
    for (size_t k = 0; k < npieces && rc == NB_OK; ++k) {
        while (nsent < npieces && nsent < k + DL_SLOTS && rc == NB_OK) {
            // the slot's earlier pieces are out
            const size_t before = nsent / DL_SLOTS;
            if (emptied[nsent % DL_SLOTS].load(std::memory_order_acquire) < before) {
                if (nsent > k) break;
                std::this_thread::yield();
                continue;
            }
            rc = send();
        }
        if (rc != NB_OK) break;
        const hipError_t e = hipEventSynchronize(b->ev[k % DL_SLOTS]);
        if (e != hipSuccess) {
            set_error("download failed: %s", hipGetErrorString(e));
            rc = NB_ERR_HIP;
            break;
        }
        if (k == 0 && npieces >= DL_SLOTS) start_workers();
        if (started > 0) {
            ready.store(k + 1, std::memory_order_release);
        } else if (got.next(p)) {
            empty(p, k);
        }
    }
    if (rc != NB_OK) stop.store(true);
    for (int t = 0; t < started; ++t) threads[t].join();
    if (rc != NB_OK) (void)hipStreamSynchronize(s);   // no copy into the block is left behind
    return rc;
}

}  // namespace

int download_fields(const DownField *f, int nf, int dev, hipStream_t s) {
    // A large array in pinned memory of the caller's takes one copy command: through
    // the pieces it would be moved twice (65536 particles 139 us against 98, 2^20
    // 1.20 ms against 0.95).  Up to a piece the command costs more (16001: 57 us
    // against 49), and nothing asks for the kind of pointer.
    unsigned todo = 0;
    for (int k = 0; k < nf; ++k) {
        if (!f[k].dst || f[k].count == 0) continue;
        if (f[k].count > DL_PIECE / sizeof(double) && runtime_memory(f[k].dst)) NB_TRY(copy_direct(f[k], s));
        else todo |= 1u << k;
    }
    size_t npieces = 0;
    Pieces it{f, nf, todo};
    Piece p;
    while (it.next(p)) ++npieces;
    if (npieces == 0) return NB_OK;
    Block *b = take_block(dev);
    if (!b) {
        for (int k = 0; k < nf; ++k)
            if (todo >> k & 1) NB_TRY(copy_direct(f[k], s));
        return NB_OK;
    }
    const int rc = copy_pieces(f, nf, todo, b, npieces, s);
    if (!g_pool.give(b)) free_block(b);
    return rc;
}

DownloadUse::DownloadUse() { g_pool.hold(); }

DownloadUse::~DownloadUse() {
    Block *b = g_pool.release();
    while (b) {
        Block *next = b->next;
        free_block(b);
        b = next;
    }
}

}  // namespace nb
