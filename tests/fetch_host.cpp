// PinnedFetch (tritify_amd/csrc/kt_fetch.h) over a runtime that queues its copies and runs them when something waits
// for them, and that fails the calls it is told to.
#include <stdint.h>
#include <stdlib.h>

#include <deque>

#include "kt_fetch.h"

namespace {

struct Op {
    void* dst;  // null: an event's mark
    const void* src;
    size_t bytes;
    int mark;
};
std::deque<Op> g_queue;
int g_marks, g_fail_kind, g_fail_at, g_calls[5], g_live;  // g_live: host blocks and events that exist
enum { ALLOC = 1, EVENT, COPY, RECORD };

bool fails(int kind) { return kind == g_fail_kind && g_calls[kind]++ >= g_fail_at; }
void run_one() {
    const Op o = g_queue.front();
    g_queue.pop_front();
    if (o.dst) memcpy(o.dst, o.src, o.bytes);
}

struct Fake {
    typedef int Err;
    typedef int Stream;
    typedef int* Event;  // the mark it was last recorded at
    static Err host_alloc(void** p, size_t n) {
        if (fails(ALLOC)) return 2;
        g_live++, *p = malloc(n);
        return 0;
    }
    static void host_free(void* p) { g_live--, free(p); }
    static Err event(Event* e) {
        if (fails(EVENT)) return 3;
        g_live++, *e = new int(0);
        return 0;
    }
    static void event_free(Event e) { g_live--, delete e; }
    static Err copy(void* d, const void* s, size_t n, Stream) {
        if (fails(COPY)) return 4;
        g_queue.push_back(Op{d, s, n, 0});
        return 0;
    }
    static Err record(Event e, Stream) {
        if (fails(RECORD)) return 5;
        *e = ++g_marks;
        g_queue.push_back(Op{nullptr, nullptr, 0, *e});
        return 0;
    }
    static Err wait(Event e) {
        while (!g_queue.empty()) {
            const bool last = g_queue.front().mark == *e;
            run_one();
            if (last) break;
        }
        return 0;
    }
    static Err drain(Stream) {
        while (!g_queue.empty()) run_one();
        return 0;
    }
};

}  // namespace

// Two calls of `bytes` each behind a kernel that is still queued when the copy is asked for; the call of kind `kind`
// fails from its `at`-th time on. Bit i of the result: call i returned success with the right bytes; bit 4: something was
// still pending when a call returned; bit 5: a block or event was left after the release; then the last error in bits 8 on.
extern "C" int fetch_case(size_t bytes, int kind, int at) {
    g_queue.clear();
    g_fail_kind = kind, g_fail_at = at, g_live = 0;
    for (int i = 0; i < 5; i++) g_calls[i] = 0;
    uint8_t *made = (uint8_t*)malloc(bytes + 1), *src = (uint8_t*)malloc(bytes + 1), *dst = (uint8_t*)malloc(bytes + 1);
    int r = 0, err = 0;
    {
        kt::PinnedFetch<Fake> f;
        for (int c = 0; c < 2; c++) {
            for (size_t i = 0; i < bytes; i++) made[i] = (uint8_t)(i * 7 + (i >> 11) + c), src[i] = 0, dst[i] = 0xEE;
            g_queue.push_back(Op{src, made, bytes, 0});  // the product, whose result the copies read
            dst[bytes] = 0x5A;
            const int e = f(dst, src, bytes, 0);
            if (e == 0 && memcmp(dst, made, bytes) == 0 && dst[bytes] == 0x5A) r |= 1 << c;
            if (e != 0) err = e;
            if (!g_queue.empty()) r |= 16;
            while (!g_queue.empty()) run_one();
        }
        f.release();
    }
    if (g_live != 0) r |= 32;
    free(made), free(src), free(dst);
    return r | err << 8;
}
extern "C" size_t fetch_block() { return kt::PinnedFetch<Fake>::BLOCK; }
