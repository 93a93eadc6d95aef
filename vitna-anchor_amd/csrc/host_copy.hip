/**
 * host_copy.hip - The device's results into a caller's memory (host_copy.h).
 * Host code only.
 *
 * A copy from the device to ordinary memory page-locks the target (or goes
 * through the runtime's own buffer) call by call, and takes the faults of a
 * fresh allocation one page at a time: 17 GB/s to touched pages, 4 GB/s to
 * fresh ones, and 32 rows of 600 KB one by one take 4.2 ms where one copy of
 * them takes 1.25. Page-locked memory takes 56 GB/s. So the rows go to
 * page-locked chunks, each with an event, and the host copies a chunk on
 * while the next one arrives, with HELPERS threads beside the caller, since
 * one thread copies 30 GB/s to touched pages and less than 10 to fresh ones
 * (32 MB: 1100 us and 3700; four threads 390 and 2500). Measured: 32 rows'
 * logits (19 MB) of a pass of 2500 us, now 2110; 4096 prefilled rows (32 MB)
 * 5100 to 6100, now 3480 with the caller's array no longer copied first.
 *
 * Small rows with gaps between them are on their way together and waited for
 * once: every second of 200 rows of 4 KB 1426 us a run at a time, now 359.
 * Memory that HIP allocated is written by the device itself: 32 rows' logits
 * into page-locked memory took 1032 us by way of the chunks and take 742.
 */

#include "host_copy.h"

#include <stdint.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>

namespace {

constexpr size_t CHUNK = 512u << 10;
constexpr int SLOTS = 32; /* 16 MB a model */
constexpr int HELPERS = 3;
/* Between the two a plain copy a row: 600 KB of one step's logits through the chunks took 2 to 40 us more (step 291 to
   296 us, token by layers 458 to 496), for the threads are not awake by then and the two chunks' events cost what the
   overlap gives. Of 4 KB the plain copy takes 8 us more (step 94, now 85), and 3 MB are level. */
constexpr size_t SMALL_BYTES = 64u << 10;
constexpr size_t HELP_BYTES = 2u << 20;
constexpr int KEPT = 512; /* a pass of 1024 rows, every second one asked for */

inline void relax() { __builtin_ia32_pause(); }

} // namespace

struct host_copy {
    char* mem;
    hipEvent_t arrived[SLOTS];
    /* the copy under way: rows row0 .. of `bytes`, `total` bytes in `chunks` chunks */
    size_t bytes, total;
    void* const* dst;
    int chunks;
    std::atomic<int> ready, claimed, copied; /* chunks in page-locked memory; taken by a thread; in place */
    std::atomic<int> slot_chunk[SLOTS];      /* the last chunk copied out of a slot */
    std::atomic<bool> closed;                /* no chunk is left to take */
    /* small runs of rows whose copies are under way, one after another in mem from its start */
    struct { size_t bytes, n; void* const* rows; } kept[KEPT];
    int n_kept;
    size_t kept_bytes;
    /* helpers */
    std::mutex m;
    std::condition_variable wake;
    int job, in_job, n_threads; /* under m */
    bool stop;
    std::thread threads[HELPERS];

    /* takes a chunk that has arrived and copies it out; false when there is none at the moment */
    bool take() {
        int i = claimed.load(std::memory_order_relaxed);
        do {
            if (i >= ready.load(std::memory_order_acquire)) return false;
        } while (!claimed.compare_exchange_weak(i, i + 1, std::memory_order_relaxed));
        const char* src = mem + (size_t)(i % SLOTS) * CHUNK;
        size_t at = (size_t)i * CHUNK;
        const size_t end = std::min(total, at + CHUNK);
        while (at < end) { /* the rows, or parts of rows, that the chunk holds */
            const size_t row = at / bytes, off = at % bytes, len = std::min(end - at, bytes - off);
            memcpy(static_cast<char*>(dst[row]) + off, src, len);
            src += len;
            at += len;
        }
        slot_chunk[i % SLOTS].store(i, std::memory_order_release);
        copied.fetch_add(1, std::memory_order_release);
        return true;
    }

    void help() {
        int seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> l(m);
                wake.wait(l, [&] { return stop || job != seen; });
                if (stop) return;
                seen = job;
                if (closed.load()) continue;
                in_job++;
            }
            while (!closed.load(std::memory_order_acquire))
                if (!take()) relax();
            std::lock_guard<std::mutex> l(m);
            in_job--;
        }
    }

    /* lets the helpers that are in the job leave it: the next one may write its fields */
    void close() {
        closed.store(true, std::memory_order_release);
        for (;;) {
            {
                std::lock_guard<std::mutex> l(m);
                if (!in_job) return;
            }
            relax();
        }
    }

    void open_helpers() {
        {
            std::lock_guard<std::mutex> l(m);
            closed.store(false);
            job++;
        }
        try {
            for (; n_threads < HELPERS; n_threads++) threads[n_threads] = std::thread([this] { help(); });
        } catch (...) { /* without them the caller copies alone */
        }
        wake.notify_all();
    }

    /* A small run of rows: on its way to mem, and from there at the next flush, so that rows with gaps between them are
       waited for once. */
    hipError_t keep(hipStream_t s, const char* dev, size_t row_bytes, size_t n, void* const* rows) {
        const size_t len = row_bytes * n;
        if (n_kept == KEPT || kept_bytes + len > CHUNK * SLOTS) {
            const hipError_t e = flush(s);
            if (e != hipSuccess) return e;
        }
        const hipError_t e = hipMemcpyAsync(mem + kept_bytes, dev, len, hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) return e;
        kept[n_kept++] = {row_bytes, n, rows};
        kept_bytes += len;
        return e;
    }

    /* (an event: hipStreamSynchronize took 4 us more a wait, a prefill of 8 rows of 512 columns 96 us and with events 87) */
    hipError_t flush(hipStream_t s) {
        if (!n_kept) return hipSuccess;
        hipError_t e = hipEventRecord(arrived[0], s);
        e = e == hipSuccess ? hipEventSynchronize(arrived[0]) : hipStreamSynchronize(s);
        const char* src = mem;
        for (int k = 0; e == hipSuccess && k < n_kept; k++)
            for (size_t r = 0; r < kept[k].n; r++, src += kept[k].bytes) memcpy(kept[k].rows[r], src, kept[k].bytes);
        n_kept = 0;
        kept_bytes = 0;
        return e;
    }

    /* what was kept is not wanted any more, but its copies write mem */
    void drop(hipStream_t s) {
        (void)hipStreamSynchronize(s);
        n_kept = 0;
        kept_bytes = 0;
    }

    hipError_t run(hipStream_t s, const char* dev, size_t row_bytes, size_t n, void* const* rows) {
        bytes = row_bytes;
        total = row_bytes * n;
        dst = rows;
        chunks = (int)((total + CHUNK - 1) / CHUNK);
        ready.store(0);
        claimed.store(0);
        copied.store(0);
        for (int i = 0; i < SLOTS; i++) slot_chunk[i].store(i - SLOTS);
        const bool helped = total >= HELP_BYTES;
        hipError_t e = hipSuccess;
        int issued = 0;
        for (int i = 0; e == hipSuccess && i < chunks; i++) {
            /* every chunk whose slot is free again; the one waited for next has to be among them */
            for (; e == hipSuccess && issued < chunks; issued++) {
                const int slot = issued % SLOTS;
                while (issued == i && slot_chunk[slot].load(std::memory_order_acquire) != issued - SLOTS)
                    if (!take()) relax();
                if (slot_chunk[slot].load(std::memory_order_acquire) != issued - SLOTS) break;
                const size_t at = (size_t)issued * CHUNK;
                e = hipMemcpyAsync(mem + (size_t)slot * CHUNK, dev + at, std::min(CHUNK, total - at), hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(arrived[slot], s);
            }
            if (e == hipSuccess) e = hipEventSynchronize(arrived[i % SLOTS]);
            if (e != hipSuccess) break;
            ready.store(i + 1, std::memory_order_release);
            if (helped && i == 0) open_helpers(); /* not before: they spin while a job is open */
            take();
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(s); /* what was issued writes mem */
        const int have = ready.load();
        while (copied.load(std::memory_order_acquire) < have)
            if (!take()) relax();
        if (helped && have) close();
        return e;
    }
};

host_copy* host_copy_create() {
    host_copy* c = new (std::nothrow) host_copy();
    if (!c) return nullptr;
    c->closed.store(true);
    bool ok = hipHostMalloc((void**)&c->mem, CHUNK * SLOTS, 0) == hipSuccess;
    for (int i = 0; ok && i < SLOTS; i++) ok = hipEventCreateWithFlags(&c->arrived[i], hipEventDisableTiming) == hipSuccess;
    if (ok) return c;
    (void)hipGetLastError();
    host_copy_destroy(c);
    return nullptr;
}

void host_copy_destroy(host_copy* c) {
    if (!c) return;
    {
        std::lock_guard<std::mutex> l(c->m);
        c->stop = true;
    }
    c->wake.notify_all();
    for (int i = 0; i < c->n_threads; i++) c->threads[i].join();
    for (int i = 0; i < SLOTS; i++)
        if (c->arrived[i]) (void)hipEventDestroy(c->arrived[i]);
    if (c->mem) (void)hipHostFree(c->mem);
    delete c;
}

/* Whether HIP allocated p: page-locked, managed or device memory, which the device copies to by itself. 0.1 us. */
static bool known(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

/* Row j follows row j - 1 of the run from i in the same 64 KB: what HIP allocates on the device begins at such a bound, so
   j is looked up no more than its neighbour was (512 rows of 4 KB would take 50 us). */
static bool beside(void* const* dst, size_t i, size_t j, size_t bytes) {
    return j > i && static_cast<char*>(dst[j]) == static_cast<char*>(dst[j - 1]) + bytes &&
           reinterpret_cast<uintptr_t>(dst[j]) >> 16 == reinterpret_cast<uintptr_t>(dst[j - 1]) >> 16;
}

hipError_t host_copy_rows(host_copy* c, hipStream_t s, const void* dev, size_t bytes, size_t n, void* const* dst) {
    hipError_t e = hipSuccess;
    bool plain = false;
    for (size_t i = 0; e == hipSuccess && i < n;) {
        const char* src = static_cast<const char*>(dev) + i * bytes;
        if (!dst[i]) { i++; continue; }
        size_t j = i; /* rows side by side on the device go as one copy, wherever each is wanted */
        while (c && j < n && dst[j] && (beside(dst, i, j, bytes) || !known(dst[j]))) j++;
        const size_t total = bytes * (j - i);
        if (j == i || (total > SMALL_BYTES && total < HELP_BYTES)) {
            j = std::max(j, i + 1);
            for (; e == hipSuccess && i < j; i++, src += bytes) e = hipMemcpyAsync(dst[i], src, bytes, hipMemcpyDeviceToHost, s);
            plain = true;
        } else if (total <= SMALL_BYTES) {
            e = c->keep(s, src, bytes, j - i, dst + i);
            i = j;
        } else {
            e = c->flush(s);
            if (e == hipSuccess) e = c->run(s, src, bytes, j - i, dst + i);
            i = j;
        }
    }
    const bool kept = c && c->n_kept;
    if (e == hipSuccess && kept) return c->flush(s);
    if (kept) c->drop(s);
    return e == hipSuccess && plain ? hipStreamSynchronize(s) : e;
}
