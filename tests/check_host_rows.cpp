// Host-only harness of the rows' way through the ring of page-locked pieces (picoforge_amd/csrc/pf_host_rows.h), built with the
// sanitizers by tests/test_host_rows.py.  A "device" is a thread that carries out the enqueued transfers one after the other,
// as a stream does, so that a piece filled or emptied before its transfer has ended is a race the thread sanitizer sees.
// Several callers, each with a ring and device rows of its own, send rows in, have the device negate them and fetch them back,
// at once: the crew is busy for some of them, and comes and goes as callers open and close.  Every 16-byte transfer must start
// on 16-byte boundaries, every row must arrive, and nothing between the rows of a pitch may be touched.
#include <stdio.h>
#include <stdlib.h>
#include <math.h>
#include <deque>
#include <functional>
#include <memory>
#include <vector>
#include "../picoforge_amd/csrc/pf_host_rows.h"

static std::atomic<int> bad{0};
static void expect(bool ok, const char *what) { if (!ok && bad++ < 10) fprintf(stderr, "%s\n", what); }

struct Device {
    std::mutex lock;
    std::condition_variable moved;
    std::deque<std::pair<unsigned long, std::function<void()>>> queue;
    unsigned long enqueued = 0, finished = 0, slot_at[PF_RING_SLOTS] = {};
    bool quit = false;
    int sends = 0, fail_at = -1;
    std::thread stream{[this] {
        std::unique_lock<std::mutex> hold(lock);
        for (;;) {
            moved.wait(hold, [&] { return quit || !queue.empty(); });
            if (queue.empty()) return;
            auto next = std::move(queue.front());
            queue.pop_front();
            hold.unlock();
            next.second();
            hold.lock();
            finished = next.first;
            moved.notify_all();
        }
    }};
    ~Device() {
        { std::lock_guard<std::mutex> hold(lock); quit = true; }
        moved.notify_all();
        stream.join();
    }
    unsigned long enqueue(std::function<void()> work) {
        std::lock_guard<std::mutex> hold(lock);
        queue.emplace_back(++enqueued, std::move(work));
        moved.notify_all();
        return enqueued;
    }
    void wait_for(unsigned long at) {
        std::unique_lock<std::mutex> hold(lock);
        moved.wait(hold, [&] { return finished >= at; });
    }
};
static int dev_bind(void *, int device) { expect(device == 3, "another device"); return 0; }
static int dev_wait(void *self, int slot) {
    Device *d = static_cast<Device *>(self);
    unsigned long at;
    { std::lock_guard<std::mutex> hold(d->lock); at = d->slot_at[slot]; }
    d->wait_for(at);
    return 0;
}
static int dev_send(void *self, int slot, void *dst, const void *src, size_t bytes, bool) {
    Device *d = static_cast<Device *>(self);
    { std::lock_guard<std::mutex> hold(d->lock); if (d->sends++ == d->fail_at) return 7; }
    if (ring_by_kernel(dst, src, bytes)) {   // 16 bytes a thread
        expect(bytes % 16 == 0, "a 16-byte transfer of another length");
        expect(((uintptr_t)dst | (uintptr_t)src) % 16 == 0, "a 16-byte transfer off a 16-byte boundary");
    }
    const unsigned long at = d->enqueue([=] { memcpy(dst, src, bytes); });
    std::lock_guard<std::mutex> hold(d->lock);
    d->slot_at[slot] = at;
    return 0;
}

struct Aligned {
    uint8_t *p;
    explicit Aligned(size_t bytes) : p((uint8_t *)aligned_alloc(256, (bytes + 255) / 256 * 256)) {}
    ~Aligned() { free(p); }
};

static void caller(int seed, int rounds) {
    unsigned state = 12345u + seed;
    auto random = [&](unsigned n) { state = state * 1664525u + 1013904223u; return (state >> 8) % n; };
    for (int round = 0; round < rounds; round++) {
        crew_retain();
        {
            Device device;
            const RingCarrier carrier = {&device, 3, dev_bind, dev_wait, dev_send};
            static const size_t widths[] = {33, 512, 510, 2560, 768};
            const size_t cols = widths[random(5)], row_bytes = 4 * cols, pitch = row_bytes + 4 * random(3);
            const size_t step = PF_RING_BYTES / row_bytes, rows = random(3) ? step * (1 + random(20)) + random((unsigned)step) : 4 * (1 + random((unsigned)(step / 4)));
            Aligned ring(PF_RING_SLOTS * PF_RING_BYTES), on_device(rows * row_bytes);
            std::vector<uint8_t> x(rows * pitch, 0xEE), y(rows * pitch, 0xDD);
            for (size_t r = 0; r < rows; r++)
                for (size_t c = 0; c < cols; c++) { const float v = (float)(random(1u << 20)) + 1.0f; memcpy(&x[r * pitch + 4 * c], &v, 4); }
            const int what = (int)random(6);   // 0: a value that is not finite in the last row; 1: a transfer fails
            if (what == 0) { const float v = round & 1 ? NAN : -INFINITY; memcpy(&x[(rows - 1) * pitch + row_bytes - 4], &v, 4); }
            RingJob in;
            in.open(carrier, ring.p, on_device.p, x.data(), pitch, row_bytes, rows);
            in.check = true;
            if (what == 1) device.fail_at = (int)random((unsigned)in.pieces);
            ring_rows_in(&in);
            expect((in.nonfinite.load() != 0) == (what == 0), "a value that is not finite");
            expect((in.error.load() == 7) == (what == 1), "the failed transfer's error");
            device.wait_for(device.enqueued);
            if (what > 1) {
                std::vector<uint8_t>().swap(x);   // the caller's rows have been read
                device.enqueue([&] { for (size_t i = 0; i < rows * cols; i++) { float v; memcpy(&v, on_device.p + 4 * i, 4); v = -v; memcpy(on_device.p + 4 * i, &v, 4); } });
                RingJob out;
                out.open(carrier, ring.p, on_device.p, y.data(), pitch, row_bytes, rows);
                const bool fine = random(8) != 0;
                CopyCrew *crew = crew_for(out);
                ring_start_out(&out, crew);
                ring_rows_out(&out, crew, fine);
                device.wait_for(device.enqueued);
                expect(out.error.load() == 0, "an error out of nothing");
                bool same = true, untouched = true;
                for (size_t r = 0; r < rows; r++) {
                    if (fine) same &= memcmp(&y[r * pitch], on_device.p + r * row_bytes, row_bytes) == 0;
                    for (size_t b = fine ? row_bytes : 0; b < pitch; b++) untouched &= y[r * pitch + b] == 0xDD;
                }
                float first;
                memcpy(&first, on_device.p, 4);
                expect(first < 0.0f, "rows that did not arrive");
                expect(same, "rows that did not come back");
                expect(untouched, "bytes that are no rows");
            }
        }
        crew_release();
    }
}

int main() {
    std::vector<std::thread> callers;
    for (int c = 0; c < 4; c++) callers.emplace_back(caller, c, 12);
    for (auto &t : callers) t.join();
    expect(g_crew == nullptr && g_crew_users == 0, "a crew nobody uses");
    printf("%d faults\n", bad.load());
    return bad.load() != 0;
}
