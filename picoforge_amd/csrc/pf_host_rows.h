// Rows between a caller's memory and the device for host-pointer forwards of longer batches: a ring of page-locked pieces and
// the threads that fill and empty them.  Nothing here knows the GPU: the pieces' transfers are calls that pf_moe_api.hip makes
// kernels and events of, and a host-side check (tests/check_host_rows.cpp) plain copies in a thread of their own.
//
// The CPU fills or empties some pieces while the others are on their way.  (A hipMemcpy2D on the caller's pageable rows moves
// them row by row, each with a wait of its own: 777 rows of 8 KB each way took 24.9 ms.)  A piece is large enough that its
// transfer hides the enqueueing.  One CPU copies at about a fifth of what the link carries, so the pieces are dealt to a few
// threads.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>

#define PF_RING_SLOTS 8
#define PF_RING_BYTES ((size_t)512 * 1024)
#define PF_CREW_HELPERS 3                            // besides the calling thread
#define PF_CREW_FROM ((size_t)1024 * 1024)           // bytes that are worth waking them for (10 to 20 us)

// The helpers, one crew for the process: started with the first workspace that takes longer batches, ended with the last.
// A call that finds the crew at work for another one copies alone.
struct CopyCrew {
    std::mutex busy, lock;
    std::condition_variable wake, done;
    std::thread thread[PF_CREW_HELPERS];
    int helpers = 0, running = 0;
    unsigned long round = 0;
    bool quit = false;
    void (*part)(void *, int, int) = nullptr;
    void *job = nullptr;
    void serve(int worker) {
        unsigned long seen = 0;
        std::unique_lock<std::mutex> hold(lock);
        for (;;) {
            wake.wait(hold, [&] { return quit || round != seen; });
            if (quit) return;
            seen = round;
            const int workers = helpers + 1;   // (the constructor has ended: the first round comes after it)
            hold.unlock();
            part(job, worker, workers);
            hold.lock();
            if (--running == 0) done.notify_one();
        }
    }
    CopyCrew() {
        for (; helpers < PF_CREW_HELPERS; helpers++) {
            try { thread[helpers] = std::thread([this, h = helpers] { serve(h + 1); }); } catch (...) { break; }
        }
    }
    ~CopyCrew() {
        { std::lock_guard<std::mutex> hold(lock); quit = true; }
        wake.notify_all();
        for (int h = 0; h < helpers; h++) thread[h].join();
    }
    // part(job, worker, workers) by every worker; the calling thread is worker 0
    void run(void (*f)(void *, int, int), void *j) {
        { std::lock_guard<std::mutex> hold(lock); part = f; job = j; running = helpers; round++; }
        wake.notify_all();
        f(j, 0, helpers + 1);
        std::unique_lock<std::mutex> hold(lock);
        done.wait(hold, [&] { return running == 0; });
    }
};
static std::mutex g_crew_lock;
static CopyCrew *g_crew = nullptr;
static int g_crew_users = 0;
static void crew_retain() {
    std::lock_guard<std::mutex> hold(g_crew_lock);
    if (g_crew_users++ == 0) g_crew = new (std::nothrow) CopyCrew();
}
static void crew_release() {
    CopyCrew *last = nullptr;
    {
        std::lock_guard<std::mutex> hold(g_crew_lock);
        if (--g_crew_users == 0) { last = g_crew; g_crew = nullptr; }
    }
    delete last;
}

// How a ring's pieces travel; the calls return 0 or an error that ends the job.
struct RingCarrier {
    void *self;
    int device;
    int (*bind)(void *self, int device);   // a helper thread is about to work for this device
    int (*wait)(void *self, int slot);     // until the slot's last transfer has ended (none yet: at once)
    int (*send)(void *self, int slot, void *dst, const void *src, size_t bytes, bool in);   // enqueues the slot's next transfer
};

// Rows between the caller's memory (a pitch) and dense device rows.  Piece p goes to worker p % workers, whose own slots its
// pieces take in turn.
struct RingJob {
    RingCarrier carrier;
    uint8_t *ring, *device;
    uint8_t *host;          // the caller's rows
    size_t pitch, row_bytes, rows, step, pieces;
    bool check;             // in: look for values that are not finite
    std::atomic<int> error, nonfinite;
    void open(const RingCarrier &c, uint8_t *pieces_at, void *device_rows, const void *host_rows, size_t host_pitch, size_t bytes, size_t count) {
        carrier = c; ring = pieces_at; device = (uint8_t *)device_rows; host = (uint8_t *)const_cast<void *>(host_rows);
        pitch = host_pitch; row_bytes = bytes; rows = count;
        step = PF_RING_BYTES / row_bytes;
        pieces = (rows + step - 1) / step;
        check = false;
        error = 0; nonfinite = 0;
    }
    size_t rows_of(size_t p) const { return rows - p * step < step ? rows - p * step : step; }
    static int slot_of(size_t p, int workers) {
        const int per = PF_RING_SLOTS / workers;
        return (int)(p % workers) * per + (int)(p / workers % per);
    }
    void fail(int e) { int none = 0; if (e) error.compare_exchange_strong(none, e); }
    void bind(int worker) { if (worker) fail(carrier.bind(carrier.self, carrier.device)); }
    void wait(int slot) { fail(carrier.wait(carrier.self, slot)); }
    void send(int slot, void *dst, const void *src, size_t bytes, bool in) { fail(carrier.send(carrier.self, slot, dst, src, bytes, in)); }
};
static inline void rows_in(void *dst, const void *src, size_t src_pitch, size_t row_bytes, size_t rows) {
    for (size_t r = 0; r < rows; r++) memcpy((uint8_t *)dst + r * row_bytes, (const uint8_t *)src + r * src_pitch, row_bytes);
}
static inline void rows_out(void *dst, size_t dst_pitch, const void *src, size_t row_bytes, size_t rows) {
    for (size_t r = 0; r < rows; r++) memcpy((uint8_t *)dst + r * dst_pitch, (const uint8_t *)src + r * row_bytes, row_bytes);
}
// whether n floats are finite: an exponent of all ones carries into the sign bit
static inline bool finite_floats(const void *p, size_t n) {
    const uint8_t *bytes = static_cast<const uint8_t *>(p);
    uint32_t carry = 0;
    for (size_t i = 0; i < n; i++) {
        uint32_t bits;
        memcpy(&bits, bytes + 4 * i, 4);
        carry |= (bits & 0x7fffffffu) + 0x00800000u;
    }
    return !(carry >> 31);
}
// Whether a transfer goes by the kernel that moves 16 bytes a thread, else by a copy.  A piece of the ring starts on a 16-byte
// boundary; a piece's device rows do not where a row is no multiple of 16 bytes.
static inline bool ring_by_kernel(const void *dst, const void *src, size_t bytes) {
    return bytes % 16 == 0 && ((uintptr_t)dst | (uintptr_t)src) % 16 == 0;
}

static inline void ring_in_part(void *job, int worker, int workers) {
    RingJob *j = static_cast<RingJob *>(job);
    j->bind(worker);
    for (size_t p = worker; p < j->pieces && !j->error.load() && !j->nonfinite.load(); p += workers) {
        const int slot = RingJob::slot_of(p, workers);
        const size_t r = p * j->step, n = j->rows_of(p);
        uint8_t *piece = j->ring + slot * PF_RING_BYTES;
        j->wait(slot);
        rows_in(piece, j->host + r * j->pitch, j->pitch, j->row_bytes, n);
        if (j->check && !finite_floats(piece, n * j->row_bytes / 4)) { j->nonfinite = 1; return; }
        j->send(slot, j->device + r * j->row_bytes, piece, n * j->row_bytes, true);
    }
}
static inline void ring_send_out(RingJob *j, size_t p, int workers) {
    const int slot = RingJob::slot_of(p, workers);
    j->send(slot, j->ring + slot * PF_RING_BYTES, j->device + p * j->step * j->row_bytes, j->rows_of(p) * j->row_bytes, false);
}
static inline void ring_out_part(void *job, int worker, int workers) {   // the first PF_RING_SLOTS pieces are on their way
    RingJob *j = static_cast<RingJob *>(job);
    j->bind(worker);
    const size_t ahead = (size_t)(PF_RING_SLOTS / workers) * workers;
    for (size_t p = worker; p < j->pieces && !j->error.load(); p += workers) {
        const int slot = RingJob::slot_of(p, workers);
        j->wait(slot);
        if (j->error.load()) break;
        rows_out(j->host + p * j->step * j->pitch, j->pitch, j->ring + slot * PF_RING_BYTES, j->row_bytes, j->rows_of(p));
        if (p + ahead < j->pieces) ring_send_out(j, p + ahead, workers);
    }
}

// The crew if the rows are worth it and it is free (its `busy` is then held), else null.
static inline CopyCrew *crew_for(const RingJob &j) {
    CopyCrew *crew = j.row_bytes * j.rows >= PF_CREW_FROM ? g_crew : nullptr;   // (a workspace with a ring keeps it alive)
    return crew && crew->helpers && PF_RING_SLOTS % (crew->helpers + 1) == 0 && crew->busy.try_lock() ? crew : nullptr;
}
// In: the caller's rows have been read, and their transfers enqueued, when this returns.
static inline void ring_rows_in(RingJob *j) {
    if (CopyCrew *crew = crew_for(*j)) { crew->run(ring_in_part, j); crew->busy.unlock(); }
    else ring_in_part(j, 0, 1);
}
// Out: the first pieces' transfers enqueued; then, where the call went well, every row into the caller's memory.  crew: from
// crew_for, given back by ring_rows_out.
static inline void ring_start_out(RingJob *j, CopyCrew *crew) {
    const int workers = crew ? crew->helpers + 1 : 1;
    for (size_t p = 0; p < j->pieces && p < PF_RING_SLOTS; p++) ring_send_out(j, p, workers);
}
static inline void ring_rows_out(RingJob *j, CopyCrew *crew, bool fine) {
    fine = fine && !j->error.load();
    if (fine && crew) crew->run(ring_out_part, j);
    else if (fine) ring_out_part(j, 0, 1);
    if (crew) crew->busy.unlock();
}
