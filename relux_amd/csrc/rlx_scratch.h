// Growable buffers of a handle: the device scratch its calls share, the
// adapter rows, and the staging slots.  Host code over an allocator the
// runtime supplies (Mem: get / put device memory, get_host / put_host pinned
// memory -- null when refused -- and sync, which waits for the handle's
// queued work), so that the rules can be tested without a device.
//
// The rules: a buffer that fits is replaced only once its successor is there,
// and a buffer whose address a captured graph may hold is never given back
// before the handle closes.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace rlx {

enum class Grow { kOk, kSync, kMemory };  // what a growth ended in

struct Scratch {
    // Scratch that calls can do without doubles up to this size; past it a
    // request gets what it asks for, not twice a large mandatory buffer.
    static constexpr size_t kOptionalDouble = (size_t)64 << 20;

    void *ptr = nullptr;
    size_t cap = 0;
    size_t peak = 0;               // largest request so far
    size_t refused = 0;            // smallest optional request the allocator refused (0: none)
    bool held = false;             // a captured graph may hold ptr
    bool reserved = false;         // sized ahead of time: optional requests do not grow it
    std::vector<void *> retired;   // superseded buffers a captured graph may hold

    // Growth to `bytes` for a call that needs them.
    template <class Mem>
    Grow need(Mem &m, size_t bytes) {
        peak = std::max(peak, bytes);
        if (bytes <= cap) return Grow::kOk;
        return grow(m, std::max(bytes, 2 * cap), bytes);
    }

    // Growth to `bytes` for a call that can do without them; false leaves the
    // buffer as it is, and a refused size is not asked for again until the
    // buffer has grown.
    template <class Mem>
    bool want(Mem &m, size_t bytes) {
        peak = std::max(peak, bytes);
        if (bytes <= cap) return true;
        if (reserved || (refused && bytes >= refused)) return false;
        const size_t n = round(std::max(bytes, std::min(2 * cap, kOptionalDouble)));
        if (!m.sync()) return false;
        void *p = m.get(n);
        if (!p) {
            refused = bytes;
            return false;
        }
        replace(m, p, n);
        return true;
    }

    // At least `bytes` from now on, and no optional growth after it.
    template <class Mem>
    Grow reserve(Mem &m, size_t bytes) {
        if (bytes > cap) {
            const Grow g = grow(m, bytes, bytes);
            if (g != Grow::kOk) return g;
        }
        reserved = true;
        return Grow::kOk;
    }

    template <class Mem>
    void release(Mem &m) {
        if (ptr) m.put(ptr);
        for (void *p : retired) m.put(p);
        retired.clear();
        ptr = nullptr;
        cap = 0;
        held = false;
    }

private:
    static size_t round(size_t n) { return (n + 65535) & ~(size_t)65535; }

    // Out of memory with the old buffer still there, that one is given up, as a
    // last resort.
    template <class Mem>
    Grow grow(Mem &m, size_t most, size_t least) {
        if (!m.sync()) return Grow::kSync;
        most = round(most);
        least = round(least);
        size_t got = most;
        void *p = m.get(got);
        if (!p && least < most) p = m.get(got = least);
        if (!p && ptr && !held) {
            m.put(ptr);
            ptr = nullptr;
            cap = 0;
            p = m.get(got = least);
        }
        if (!p) return Grow::kMemory;
        replace(m, p, got);
        return Grow::kOk;
    }

    template <class Mem>
    void replace(Mem &m, void *p, size_t n) {
        if (ptr && held)
            retired.push_back(ptr);
        else if (ptr)
            m.put(ptr);
        ptr = p;
        cap = n;
        refused = 0;
        held = false;
    }
};

// A staging slot's pair of buffers (pinned host, device) of one capacity.
struct StagePair {
    void *host = nullptr;
    void *dev = nullptr;
    size_t cap = 0;

    // Growth to `bytes`; on failure the pair there was stays.
    template <class Mem>
    Grow grow(Mem &m, size_t bytes) {
        if (bytes <= cap) return Grow::kOk;
        // The device copy may still be read by queued kernels.
        if (!m.sync()) return Grow::kSync;
        const size_t n = (bytes + 4095) & ~(size_t)4095;
        void *h = m.get_host(n), *d = h ? m.get(n) : nullptr;
        if (!d) {
            if (h) m.put_host(h);
            return Grow::kMemory;
        }
        release(m);
        host = h;
        dev = d;
        cap = n;
        return Grow::kOk;
    }

    template <class Mem>
    void release(Mem &m) {
        if (host) m.put_host(host);
        if (dev) m.put(dev);
        host = dev = nullptr;
        cap = 0;
    }
};

}  // namespace rlx
