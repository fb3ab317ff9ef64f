// fm_copy.hip -- large transfers between device staging and the caller's (pageable) host arrays.
//
// A copy to pageable memory runs at the speed of one host thread that also takes the page faults of
// the caller's fresh arrays (72 MB, the state of 1,048,576 molecules: 8 ms).  Here the data passes
// through pinned slots: the calling thread queues the device copies in order, and a few threads move
// each slot to or from the caller's memory as it is ready (the same 72 MB: 3.7 ms, of which the link takes most).
//
// The pinned memory belongs to a pool of the process: a transfer borrows a set and gives it back before
// it returns, at most POOL_SETS exist (of up to 24 MiB each, as much as a transfer has needed), and the
// pool is freed with the last context.  Downloads make and grow the sets, uploads use what is there.  A
// transfer that finds no set, or no thread, is done by the plain copy.
//
// Slots of 4 MiB where there are enough of them for the threads: in the first 15 ms after a context is made
// the device takes about 170 us for 2 MiB and 230 for 4, however the copies are queued (55 and 105 later
// on), so the first reading of 1,048,576 molecules took 8.2 ms in slots of 2 MiB, by the plain copy 5.9 and
// in slots of 4 MiB 5.8; later ones 2.07, 4.24 and 1.87 ms.  7.8 MB take 340 us in slots of 2 MiB, 370 in
// slots of 4.
#include "fm_internal.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <exception>
#include <new>
#include <thread>
#include <vector>

#define UNIT_BYTES (2u << 20)  // a slot is one or two of these
#define NUNITS 12
#define TWO_UNITS (24u << 20)  // two from this size on
#define POOL_SETS 4
#define COPY_THREADS 6
#define COPY_SEGS 4          // segments of a call
// Below these the threads cost more than they save.  Us by the plain copy and through the slots: to the
// host 4.5 MB 290 and 240, 7.8 MB 480 and 340; to the device 4.5 MB 197 and 240, 12.3 MB 475 and 470, 24 MB
// from the arrays of the transfer before 715 and 770, 30 MB 920 and 870, 37 MB 1,400 and 1,020 (from new
// arrays the slots gain from 13 MB on)
#define COPY_MIN_HOST (4u << 20)
#define COPY_MIN_DEVICE (24u << 20)

namespace {

struct SlotSet {
    char* p = nullptr;           // n x UNIT_BYTES, pinned
    hipEvent_t ev[NUNITS] = {};  // the device copy of each slot
    int n = 0;
    int dev = -1;
    bool busy = false;
};

std::mutex g_mu;
SlotSet* g_sets[POOL_SETS] = {};
int g_contexts = 0;

void free_set(SlotSet* s) {
    for (hipEvent_t e : s->ev)
        if (e) hipEventDestroy(e);
    if (s->p) hipHostFree(s->p);
    delete s;
}

// a set of fewer units than wanted gets that many, in one allocation (six take 1.5 ms longer to free); if
// they cannot be had it keeps what it has
void grow_set(SlotSet* s, int want) {
    if (s->n >= want) return;
    char* p = nullptr;
    bool ok = hipHostMalloc((void**)&p, (size_t)want * UNIT_BYTES, hipHostMallocDefault) == hipSuccess;
    for (int k = 0; ok && k < want; ++k)
        ok = s->ev[k] || hipEventCreateWithFlags(&s->ev[k], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
    } else {
        std::swap(p, s->p);
        s->n = want;
    }
    if (p) hipHostFree(p);
}

// a set with at least one unit, `want` of them if they can be had; without `grow` a set of that many or none
// (the pinned memory costs 2 ms, more than an upload of a context's only state gains by it)
SlotSet* borrow(int dev, int want, bool grow) {
    std::lock_guard<std::mutex> lock(g_mu);
    SlotSet** room = nullptr;
    for (SlotSet*& s : g_sets) {
        if (!s) room = &s;
        else if (!s->busy && s->dev == dev && (grow || s->n >= want)) {
            grow_set(s, want);
            s->busy = true;
            return s;
        }
    }
    if (!room || !grow) return nullptr;
    SlotSet* s = new (std::nothrow) SlotSet();
    if (!s) return nullptr;
    s->dev = dev;
    grow_set(s, want);
    if (s->n == 0) {
        free_set(s);
        return nullptr;
    }
    s->busy = true;
    *room = s;
    return s;
}

void give_back(SlotSet* s) {
    std::lock_guard<std::mutex> lock(g_mu);
    s->busy = false;
}

struct Chunk {
    char *host, *dev;
    size_t n;
};

int plain_copy(fm_ctx* c, const CopySeg* seg, int nseg, bool to_host) {
    for (int k = 0; k < nseg; ++k)
        if (seg[k].host && seg[k].bytes) {
            if (to_host) FM_HIP(hipMemcpyAsync(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost, c->stream));
            else FM_HIP(hipMemcpyAsync(seg[k].dev, seg[k].host, seg[k].bytes, hipMemcpyHostToDevice, c->stream));
        }
    return 0;
}

// Memory that the runtime knows (pinned, managed or a device's): the device copies it by itself, at the
// link's rate (72 MB, the state of 1,048,576 molecules: 1.40 ms; through the slots 2.04), and a thread
// here may not be able to touch it.
bool runtime_memory(const void* p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

// One transfer.  issued: chunks whose device copy is queued (their slot's event recorded); moved[i]:
// chunk i's host side is done; failed: a HIP call failed, everyone stops.
struct Transfer {
    fm_ctx* c;
    SlotSet* s;
    std::vector<Chunk> ch;
    bool to_host;
    size_t slot_bytes, ring;     // and slots in use
    std::atomic<size_t> next{0}, issued{0};
    std::vector<std::atomic<char>> moved;
    std::atomic<int> failed{0};
    explicit Transfer(size_t n) : moved(n) {
        for (auto& m : moved) m.store(0, std::memory_order_relaxed);
    }

    bool until_issued(size_t n) {
        while (issued.load(std::memory_order_acquire) < n) {
            if (failed.load(std::memory_order_relaxed)) return false;
            std::this_thread::yield();
        }
        return true;
    }
    bool until_moved(size_t i) {
        while (!moved[i].load(std::memory_order_acquire)) {
            if (failed.load(std::memory_order_relaxed)) return false;
            std::this_thread::yield();
        }
        return true;
    }
    bool device_done(size_t slot) {
        if (hipEventSynchronize(s->ev[slot]) == hipSuccess) return true;
        failed.store(1);
        return false;
    }

    // a worker: the host side of one chunk after another
    void work() {
        if (hipSetDevice(c->dev) != hipSuccess) {
            failed.store(1);
            return;
        }
        for (;;) {
            const size_t i = next.fetch_add(1);
            if (i >= ch.size()) return;
            const size_t slot = i % ring;
            char* pin = s->p + slot * slot_bytes;
            if (to_host) {
                if (!until_issued(i + 1) || !device_done(slot)) return;
                memcpy(ch[i].host, pin, ch[i].n);
            } else {
                // (the slot's copy of `ring` chunks ago has left it)
                if (i >= ring && (!until_issued(i - ring + 1) || !device_done(slot))) return;
                memcpy(pin, ch[i].host, ch[i].n);
            }
            moved[i].store(1, std::memory_order_release);
        }
    }

    // the calling thread: the device side in order
    bool issue() {
        for (size_t i = 0; i < ch.size(); ++i) {
            const size_t slot = i % ring;
            char* pin = s->p + slot * slot_bytes;
            if (to_host ? (i >= ring && !until_moved(i - ring)) : !until_moved(i)) return false;
            const hipError_t e = to_host
                                     ? hipMemcpyAsync(pin, ch[i].dev, ch[i].n, hipMemcpyDeviceToHost, c->stream)
                                     : hipMemcpyAsync(ch[i].dev, pin, ch[i].n, hipMemcpyHostToDevice, c->stream);
            if (e != hipSuccess || hipEventRecord(s->ev[slot], c->stream) != hipSuccess) {
                failed.store(1);
                return false;
            }
            issued.store(i + 1, std::memory_order_release);
        }
        return true;
    }
};

}  // namespace

void copy_pool_retain() {
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_contexts;
}

void copy_pool_release() {
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_contexts > 0) return;
    for (SlotSet*& s : g_sets) {
        if (s) free_set(s);
        s = nullptr;
    }
}

// Copies the segments between the device and the host, in stream order.  Host data is in place (to the
// device: no longer needed) when it returns, unless the transfer is small: then after the stream's
// next synchronisation, which every caller does.
int copy_segments(fm_ctx* c, const CopySeg* all, int n_all, bool to_host) {
    size_t total = 0;
    for (int k = 0; k < n_all; ++k) total += all[k].host ? all[k].bytes : 0;
    const size_t least = to_host ? COPY_MIN_HOST : COPY_MIN_DEVICE;
    if (total < least) return plain_copy(c, all, n_all, to_host);
    CopySeg seg[COPY_SEGS];
    int nseg = 0;
    total = 0;
    for (int k = 0; k < n_all; ++k) {
        if (!all[k].host || !all[k].bytes) continue;
        if (n_all > COPY_SEGS || runtime_memory(all[k].host)) {
            if (int rc = plain_copy(c, all + k, 1, to_host)) return rc;
        } else {
            seg[nseg++] = all[k];
            total += all[k].bytes;
        }
    }
    if (total < least) return plain_copy(c, seg, nseg, to_host);
    SlotSet* s = borrow(c->dev, (int)std::min<size_t>(NUNITS, total / UNIT_BYTES + 2), to_host);
    if (!s) return plain_copy(c, seg, nseg, to_host);
    const size_t slot_bytes = total >= TWO_UNITS && s->n >= 2 ? 2 * UNIT_BYTES : UNIT_BYTES;
    int rc = 0;
    std::vector<std::thread> th;
    try {
        std::vector<Chunk> ch;
        for (int k = 0; k < nseg; ++k)
            for (size_t o = 0; seg[k].host && o < seg[k].bytes;) {
                // (chunks end where the host's 2 MiB pages do: no two threads take the fault of one page)
                char* h = (char*)seg[k].host + o;
                const size_t n = std::min<size_t>(slot_bytes - ((uintptr_t)h & (slot_bytes - 1)), seg[k].bytes - o);
                ch.push_back({h, (char*)seg[k].dev + o, n});
                o += n;
            }
        Transfer t(ch.size());
        t.c = c;
        t.s = s;
        t.ch.swap(ch);
        t.to_host = to_host;
        t.slot_bytes = slot_bytes;
        t.ring = (size_t)s->n * UNIT_BYTES / slot_bytes;
        const size_t want = std::min<size_t>(COPY_THREADS, t.ch.size() / 2);
        th.reserve(want);
        try {
            while (th.size() < want) th.emplace_back([&t] { t.work(); });
        } catch (const std::exception&) {  // fewer threads, or none
        }
        if (th.empty()) {
            rc = plain_copy(c, seg, nseg, to_host);
        } else {
            const bool ok = t.issue();
            for (auto& x : th) x.join();
            // (a slot is lent again only after its last device copy)
            const hipError_t e = hipStreamSynchronize(c->stream);
            if (!ok || t.failed.load() || e != hipSuccess) rc = fm_set_error(FM_EHIP, "staged host copy failed: %s", hipGetErrorString(e));
        }
    } catch (const std::bad_alloc&) {  // (before any thread started)
        rc = plain_copy(c, seg, nseg, to_host);
    }
    give_back(s);
    return rc;
}
