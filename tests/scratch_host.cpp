// Scenarios of the growable buffers (relux_amd/csrc/rlx_scratch.h) over an
// allocator that counts, remembers what is alive and refuses on demand.
// usage: scratch_host SCENARIO; exit status 0: it holds.
#include "rlx_scratch.h"

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

using rlx::Grow;
using rlx::Scratch;
using rlx::StagePair;

struct Mem {
    std::map<void *, size_t> live, host;
    size_t limit = (size_t)1 << 40;  // device bytes that may be alive at once
    bool host_ok = true, sync_ok = true;
    int gets = 0, puts = 0, syncs = 0;
    uintptr_t next = 0x1000;
    size_t used() const {
        size_t n = 0;
        for (auto &p : live) n += p.second;
        return n;
    }
    void *get(size_t n) {
        gets++;
        if (used() + n > limit) return nullptr;
        void *p = (void *)(next += 0x1000);
        live[p] = n;
        return p;
    }
    void put(void *p) {
        puts++;
        if (!live.erase(p)) std::abort();  // not alive: freed twice
    }
    void *get_host(size_t n) {
        if (!host_ok) return nullptr;
        void *p = (void *)(next += 0x1000);
        host[p] = n;
        return p;
    }
    void put_host(void *p) {
        if (!host.erase(p)) std::abort();
    }
    bool sync() {
        syncs++;
        return sync_ok;
    }
};

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s\n", __LINE__, #x);              \
            return 1;                                                \
        }                                                            \
    } while (0)

constexpr size_t MB = (size_t)1 << 20;

// The address a captured graph holds stays allocated through every growth,
// and goes with the handle.
static int held() {
    for (int how = 0; how < 3; how++) {
        Mem m;
        Scratch s;
        CHECK(s.need(m, 3 * MB) == Grow::kOk);
        void *graph = s.ptr;
        s.held = true;
        CHECK(how == 0 ? s.need(m, 9 * MB) == Grow::kOk : how == 1 ? s.want(m, 9 * MB)
                                                                 : s.reserve(m, 9 * MB) == Grow::kOk);
        CHECK(s.ptr != graph && s.cap >= 9 * MB);
        CHECK(m.live.count(graph) && m.live[graph] >= 3 * MB);
        // the new buffer is in no graph: it goes when it is outgrown
        void *second = s.ptr;
        CHECK(s.need(m, 100 * MB) == Grow::kOk);
        CHECK(m.live.count(graph) && !m.live.count(second));
        s.release(m);
        CHECK(m.live.empty());
    }
    // out of memory: a held buffer is not the one to give up
    Mem m;
    Scratch s;
    CHECK(s.need(m, 3 * MB) == Grow::kOk);
    s.held = true;
    void *graph = s.ptr;
    m.limit = 6 * MB;
    CHECK(s.need(m, 5 * MB) == Grow::kMemory);
    CHECK(s.ptr == graph && s.cap >= 3 * MB && m.live.count(graph));
    return 0;
}

// A refused optional growth leaves the buffer, and is not tried again until
// the buffer has grown.
static int refused() {
    Mem m;
    Scratch s;
    CHECK(s.need(m, 10 * MB) == Grow::kOk);
    void *p = s.ptr;
    m.limit = 40 * MB;
    CHECK(!s.want(m, 64 * MB));
    CHECK(s.ptr == p && s.cap == 10 * MB && m.live.count(p) && m.puts == 0);
    const int gets = m.gets, syncs = m.syncs;
    CHECK(!s.want(m, 64 * MB) && !s.want(m, 70 * MB));
    CHECK(m.gets == gets && m.syncs == syncs);
    CHECK(s.want(m, 5 * MB) && s.ptr == p);  // (fits)
    CHECK(s.want(m, 20 * MB) && s.cap >= 20 * MB && !m.live.count(p));
    m.limit = 400 * MB;
    CHECK(s.want(m, 64 * MB));
    CHECK(s.peak == 70 * MB);
    return 0;
}

// An optional request behind a large mandatory buffer asks for what it needs.
static int no_doubling() {
    Mem m;
    Scratch s;
    CHECK(s.need(m, 3000 * MB) == Grow::kOk);
    CHECK(s.want(m, 3064 * MB));
    CHECK(s.cap == 3064 * MB);
    Scratch t;
    CHECK(t.want(m, 20 * MB) && t.want(m, 21 * MB) && t.cap == 40 * MB);  // small ones double
    CHECK(t.want(m, 41 * MB) && t.cap == 64 * MB);
    // mandatory growth doubles, as a context that grows call by call needs
    CHECK(t.need(m, 65 * MB) == Grow::kOk && t.cap == 128 * MB);
    return 0;
}

// Mandatory growth in a memory that holds no two buffers at once still works.
static int last_resort() {
    Mem m;
    Scratch s;
    CHECK(s.need(m, 30 * MB) == Grow::kOk);
    m.limit = 50 * MB;
    CHECK(s.need(m, 40 * MB) == Grow::kOk);
    CHECK(s.cap == 40 * MB && m.live.size() == 1);
    CHECK(s.need(m, 60 * MB) == Grow::kMemory);
    CHECK(s.cap == 0 && !s.ptr && m.live.empty());
    CHECK(s.need(m, 10 * MB) == Grow::kOk);
    m.sync_ok = false;
    void *p = s.ptr;
    CHECK(s.need(m, 20 * MB) == Grow::kSync && s.ptr == p && s.cap == 10 * MB);
    CHECK(!s.want(m, 20 * MB) && s.ptr == p);
    return 0;
}

// A reserved buffer does not grow for an optional request; it still counts it.
static int reserved() {
    Mem m;
    Scratch s;
    CHECK(s.want(m, MB));
    CHECK(s.reserve(m, 8 * MB) == Grow::kOk && s.cap == 8 * MB && s.peak == MB);
    const int gets = m.gets;
    CHECK(s.want(m, 8 * MB) && !s.want(m, 9 * MB) && m.gets == gets);
    CHECK(s.peak == 9 * MB);
    CHECK(s.need(m, 10 * MB) == Grow::kOk);  // (a call that needs it)
    CHECK(s.reserve(m, 2 * MB) == Grow::kOk && s.cap >= 10 * MB);
    m.limit = 0;
    const size_t cap = s.cap;
    s.held = true;
    CHECK(s.reserve(m, 100 * MB) == Grow::kMemory && s.cap == cap && s.ptr);
    Scratch none;  // calls that need no workspace reserve none
    CHECK(none.reserve(m, 0) == Grow::kOk && !none.want(m, MB) && none.cap == 0);
    return 0;
}

// A staging slot whose growth fails keeps its pair and the capacity that goes
// with it; the next plans that fit are copied into live buffers.
static int stage() {
    Mem m;
    StagePair s;
    CHECK(s.grow(m, 65536) == Grow::kOk && s.cap == 65536);
    void *h = s.host, *d = s.dev;
    m.limit = 65536;  // the device half
    CHECK(s.grow(m, 200000) == Grow::kMemory);
    CHECK(s.host == h && s.dev == d && s.cap == 65536 && m.host.count(h) && m.live.count(d));
    CHECK(m.host.size() == 1);
    m.limit = 10 * MB;
    m.host_ok = false;  // the pinned half
    CHECK(s.grow(m, 200000) == Grow::kMemory && s.host == h && s.dev == d && s.cap == 65536);
    m.host_ok = true;
    CHECK(s.grow(m, 200000) == Grow::kOk && s.cap >= 200000 && !m.host.count(h) && !m.live.count(d));
    s.release(m);
    CHECK(m.host.empty() && m.live.empty() && s.cap == 0);
    // a first growth that fails leaves nothing to copy into, and says so
    StagePair e;
    m.limit = 0;
    CHECK(e.grow(m, 100) == Grow::kMemory && e.cap == 0 && !e.host && m.host.empty());
    return 0;
}

int main(int argc, char **argv) {
    const struct {
        const char *name;
        int (*run)();
    } all[] = {{"held", held},         {"refused", refused},   {"no_doubling", no_doubling},
               {"last_resort", last_resort}, {"reserved", reserved}, {"stage", stage}};
    for (auto &t : all)
        if (argc > 1 && !std::strcmp(argv[1], t.name)) return t.run();
    return 2;
}
