// Rows between a caller's memory and the device for host-pointer forwards of longer batches: a ring of page-locked pieces and
// the threads that fill and empty them.  Nothing here knows the GPU: the pieces' transfers are calls that pf_moe_api.hip makes
// kernels and events of, and a host-side check (tests/check_host_rows.cpp) plain copies in a thread of their own.
//
// The CPU fills or empties some pieces while the others are on their way.  (A hipMemcpy2D on the caller's pageable rows moves
// them row by row, each with a wait of its own: 777 rows of 8 KB each way took 24.9 ms.)  A piece is large enough that its
// transfer hides the enqueueing.  One CPU copies at about a fifth of what the link carries, so a few threads share the copying,
// and they share every piece: parts of it go to whoever is free, in order.  (With whole pieces dealt to the threads the first
// transfer started, and the last piece's copy ended, when one thread had copied 512 KB, 55 us each.)  A piece is a quarter of
// the rows, between 256 KB and 1 MB: a kernel moves 512 KB at 35 GB/s, 1 MB at 38 in and 44 out, all of 6 MB at 42 and 51, and
// the first piece's copy and the last one's hide behind nothing.  A call of 777 rows of 8 KB 706 -> 686 us, with pieces of
// 512 KB 696; calls of 300 rows with pieces of 256 KB 472, of a quarter 432.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>

#define PF_RING_SLOTS 4                              // (8, twice the page-locked memory: 777 rows of 8 KB and 1024 of 10 KB take the same time)
#define PF_RING_BYTES ((size_t)1024 * 1024)          // a piece at most
#define PF_RING_PARTS 16                             // of a piece, each copied by one thread
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

// Rows between the caller's memory (a pitch) and dense device rows.  Piece p has slot p % PF_RING_SLOTS; its parts are handed
// out in order, piece after piece, and who ends a piece's last part sends it (in) or the slot's next one (out).
struct RingJob {
    RingCarrier carrier;
    uint8_t *ring, *device;
    uint8_t *host;          // the caller's rows
    size_t pitch, row_bytes, rows, step, pieces;
    bool check;             // in: look for values that are not finite
    std::atomic<int> error, nonfinite;
    std::atomic<size_t> next;                                       // part to hand out
    std::atomic<size_t> sent[PF_RING_SLOTS], ended[PF_RING_SLOTS];  // a slot's pieces that have been sent; its parts that have been copied
    void open(const RingCarrier &c, uint8_t *pieces_at, void *device_rows, const void *host_rows, size_t host_pitch, size_t bytes, size_t count) {
        carrier = c; ring = pieces_at; device = (uint8_t *)device_rows; host = (uint8_t *)const_cast<void *>(host_rows);
        pitch = host_pitch; row_bytes = bytes; rows = count;
        const size_t quarter = rows * row_bytes / 4, least = PF_RING_BYTES / 4;
        const size_t bytes_a_piece = quarter < least ? least : quarter < PF_RING_BYTES ? quarter : PF_RING_BYTES;
        step = (row_bytes <= bytes_a_piece ? bytes_a_piece : PF_RING_BYTES) / row_bytes;
        pieces = (rows + step - 1) / step;
        check = false;
        error = 0; nonfinite = 0; next = 0;
        for (int s = 0; s < PF_RING_SLOTS; s++) { sent[s] = 0; ended[s] = 0; }
    }
    size_t rows_of(size_t p) const { return rows - p * step < step ? rows - p * step : step; }
    static int slot_of(size_t p) { return (int)(p % PF_RING_SLOTS); }
    bool stopped() const { return error.load() != 0 || nonfinite.load() != 0; }
    void fail(int e) { int none = 0; if (e) error.compare_exchange_strong(none, e); }
    void bind(int worker) { if (worker) fail(carrier.bind(carrier.self, carrier.device)); }
    void send(size_t p, bool in) {
        const int slot = slot_of(p);
        uint8_t *piece = ring + slot * PF_RING_BYTES, *there = device + p * step * row_bytes;
        fail(carrier.send(carrier.self, slot, in ? there : piece, in ? piece : there, rows_of(p) * row_bytes, in));
        sent[slot].fetch_add(1);
    }
    // The next part: of piece p, rows [first, last) of it; false when there is none left or the job has stopped.
    struct Part { size_t p, first, last; };
    bool take(Part *part) {
        const size_t q = next.fetch_add(1), share = (step + PF_RING_PARTS - 1) / PF_RING_PARTS;
        part->p = q / PF_RING_PARTS;
        if (part->p >= pieces || stopped()) return false;
        const size_t n = rows_of(part->p), from = q % PF_RING_PARTS * share;
        part->first = from < n ? from : n;
        part->last = from + share < n ? from + share : n;
        return true;
    }
    // Until `count` pieces have been sent through the slot and the last of them has arrived; false when the job stops.  (The
    // parts before this one are all in other threads' hands, so the piece is sent without this thread.)
    bool await(int slot, size_t count) {
        while (sent[slot].load() < count) {
            if (stopped()) return false;
            std::this_thread::yield();
        }
        fail(carrier.wait(carrier.self, slot));
        return !stopped();
    }
    bool ends_piece(size_t p) { return ended[slot_of(p)].fetch_add(1) + 1 == PF_RING_PARTS * (p / PF_RING_SLOTS + 1); }
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

static inline void ring_in_part(void *job, int worker, int) {
    RingJob *j = static_cast<RingJob *>(job);
    j->bind(worker);
    for (RingJob::Part t; j->take(&t);) {
        const int slot = RingJob::slot_of(t.p);
        uint8_t *to = j->ring + slot * PF_RING_BYTES + t.first * j->row_bytes;
        if (!j->await(slot, t.p / PF_RING_SLOTS)) return;
        rows_in(to, j->host + (t.p * j->step + t.first) * j->pitch, j->pitch, j->row_bytes, t.last - t.first);
        if (j->check && !finite_floats(to, (t.last - t.first) * j->row_bytes / 4)) { j->nonfinite = 1; return; }
        if (j->ends_piece(t.p)) j->send(t.p, true);
    }
}
static inline void ring_out_part(void *job, int worker, int) {   // the first PF_RING_SLOTS pieces are on their way
    RingJob *j = static_cast<RingJob *>(job);
    j->bind(worker);
    for (RingJob::Part t; j->take(&t);) {
        const int slot = RingJob::slot_of(t.p);
        if (!j->await(slot, t.p / PF_RING_SLOTS + 1)) return;
        rows_out(j->host + (t.p * j->step + t.first) * j->pitch, j->pitch, j->ring + slot * PF_RING_BYTES + t.first * j->row_bytes, j->row_bytes,
                 t.last - t.first);
        if (j->ends_piece(t.p) && t.p + PF_RING_SLOTS < j->pieces) j->send(t.p + PF_RING_SLOTS, false);
    }
}

// The crew if the rows are worth it and it is free (its `busy` is then held), else null.
static inline CopyCrew *crew_for(const RingJob &j) {
    CopyCrew *crew = j.row_bytes * j.rows >= PF_CREW_FROM ? g_crew : nullptr;   // (a workspace with a ring keeps it alive)
    return crew && crew->helpers && crew->busy.try_lock() ? crew : nullptr;
}
// In: the caller's rows have been read, and their transfers enqueued, when this returns.
static inline void ring_rows_in(RingJob *j) {
    if (CopyCrew *crew = crew_for(*j)) { crew->run(ring_in_part, j); crew->busy.unlock(); }
    else ring_in_part(j, 0, 1);
}
// Out: the first pieces' transfers enqueued; then, where the call went well, every row into the caller's memory.  crew: from
// crew_for, given back by ring_rows_out.
static inline void ring_start_out(RingJob *j, CopyCrew *) {
    for (size_t p = 0; p < j->pieces && p < PF_RING_SLOTS; p++) j->send(p, false);
}
static inline void ring_rows_out(RingJob *j, CopyCrew *crew, bool fine) {
    fine = fine && !j->error.load();
    if (fine && crew) crew->run(ring_out_part, j);
    else if (fine) ring_out_part(j, 0, 1);
    if (crew) crew->busy.unlock();
}
