// xfer.hpp -- grids between the host heap (the reference's AoS FP64 arrays,
// component fastest) and the device (structure of arrays, storage precision).
//
// A transfer runs through a small ring of pinned slots: host memcpy to or from
// a slot on one side, a kernel that reads or writes the slot over PCIe and
// transposes on the way on the other, so that a grid crosses in one launch and
// without a device staging array.  The ring is kept by its owner (one per
// library context, XFER_SLOTS x XFER_SLOT_BYTES of pinned memory, released with
// the context): pinning memory for every call cost more than the transfer
// (400 MB of grids: 100 ms, of which the PCIe time is 7 ms at 57 GB/s).
//
// Transfers of XFER_THREADED bytes or more copy on the host with a few threads
// of their own while the calling thread launches; one thread moves about 10
// GB/s, PCIe five times that.  All HIP calls stay on the calling thread.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace amrgpu {

// A grid on the device: element offset of component 0, component stride, and
// its first cell in the transfer's cell numbering (cells grid by grid, ghost
// cells included, in storage order).
struct XferGrid {
    int64_t off, plane, cell0;
};

// Elements [e0, e1) of a transfer (cell * nv + component) between the slot
// `stage` and the grids; `grids` null: the one grid `one`.  dst2: a second
// array that receives the same values (to the device only), or null.
struct XferArgs {
    double* stage;
    const XferGrid* grids;
    XferGrid one;
    void* data;
    void* data2;
    int64_t e0, e1;
    int32_t ngrids, nv;
};
hipError_t launch_xfer(bool to_dev, int esize, const XferArgs& a, hipStream_t st);

constexpr int XFER_SLOTS = 8;
constexpr size_t XFER_SLOT_BYTES = 2u << 20;
constexpr size_t XFER_THREADED = 8u << 20;
constexpr int XFER_WORKERS = 6;

class XferRing {
    char* base_ = nullptr;
    hipEvent_t ev_[XFER_SLOTS] = {};
    bool busy_[XFER_SLOTS] = {};   // a kernel may still read the slot
    int next_ = 0;

    hipError_t ensure() {
        if (base_) return hipSuccess;
        hipError_t e = hipHostMalloc((void**)&base_, XFER_SLOTS * XFER_SLOT_BYTES, hipHostMallocDefault);
        for (int s = 0; s < XFER_SLOTS && e == hipSuccess; s++)
            e = hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming);
        if (e != hipSuccess) release();
        return e;
    }
    double* slot(int s) { return reinterpret_cast<double*>(base_ + s * XFER_SLOT_BYTES); }
    hipError_t free_slot(int s) {
        if (!busy_[s]) return hipSuccess;
        hipError_t e = hipEventSynchronize(ev_[s]);
        busy_[s] = e != hipSuccess;
        return e;
    }

public:
    void release() {
        for (int s = 0; s < XFER_SLOTS; s++) {
            if (busy_[s]) hipEventSynchronize(ev_[s]);
            if (ev_[s]) hipEventDestroy(ev_[s]);
            ev_[s] = nullptr;
            busy_[s] = false;
        }
        if (base_) hipHostFree(base_);
        base_ = nullptr;
        next_ = 0;
    }

    // Moves elements [0, total) of the transfer described by `a` (stage and
    // e0, e1 are set here).  host(e0, e1, slot): the host side of elements
    // [e0, e1), called for disjoint ranges and possibly from several threads.
    // To the device: returns when the host data has been read; the kernels are
    // queued on the stream.  To the host: returns with the data there.
    template <class Host>
    hipError_t run(bool to_dev, int esize, XferArgs a, int64_t total, hipStream_t st, Host host) {
        if (total <= 0) return hipSuccess;
        hipError_t e = ensure();
        if (e != hipSuccess) return e;
        const int64_t per = XFER_SLOT_BYTES / sizeof(double);
        const int64_t n = (total + per - 1) / per;
        const int first = next_;
        next_ = (int)((first + n) % XFER_SLOTS);
        auto slot_of = [&](int64_t k) { return (int)((first + k) % XFER_SLOTS); };
        auto lo = [&](int64_t k) { return k * per; };
        auto hi = [&](int64_t k) { return std::min(total, (k + 1) * per); };
        auto launch = [&](int64_t k) {
            const int s = slot_of(k);
            a.stage = slot(s);
            a.e0 = lo(k);
            a.e1 = hi(k);
            hipError_t r = launch_xfer(to_dev, esize, a, st);
            if (r == hipSuccess) r = hipEventRecord(ev_[s], st);
            busy_[s] = r == hipSuccess;
            return r;
        };
        int nw = 0;
        if ((size_t)total * sizeof(double) >= XFER_THREADED)
            nw = std::min<int>(XFER_WORKERS, (int)std::thread::hardware_concurrency() / 2);
        if (nw < 2) return serial(to_dev, n, slot_of, lo, hi, launch, host);

        // every slot free, then the calling thread launches and waits for
        // events while the workers do the host side, LAG slots behind (to the
        // host) or ahead of it
        for (int s = 0; s < XFER_SLOTS; s++)
            if ((e = free_slot(s)) != hipSuccess) return e;
        constexpr int LAG = XFER_SLOTS / 2;
        std::atomic<int64_t> take{0}, gate{to_dev ? XFER_SLOTS : 0};   // chunks the workers may touch
        std::atomic<bool> stop{false};
        std::vector<std::atomic<char>> done(n);                        // host side finished
        for (auto& d : done) d.store(0, std::memory_order_relaxed);
        auto work = [&] {
            for (;;) {
                const int64_t k = take.fetch_add(1);
                if (k >= n) return;
                while (gate.load(std::memory_order_acquire) <= k) {
                    if (stop.load(std::memory_order_relaxed)) return;
                    std::this_thread::yield();
                }
                host(lo(k), hi(k), slot(slot_of(k)));
                done[k].store(1, std::memory_order_release);
            }
        };
        auto wait_done = [&](int64_t k) {
            while (!done[k].load(std::memory_order_acquire)) std::this_thread::yield();
        };
        std::vector<std::thread> pool;
        pool.reserve(nw);
        try {
            for (int t = 0; t < nw; t++) pool.emplace_back(work);
        } catch (const std::system_error&) {
            // fewer threads than asked for; with none the calling thread does it all
            if (pool.empty()) return serial(to_dev, n, slot_of, lo, hi, launch, host);
        }
        for (int64_t k = 0; k < n + LAG && e == hipSuccess; k++) {
            if (k >= LAG && (k - LAG < n)) {
                // the kernel of chunk k - LAG has run: its slot can be refilled
                // (to the device) or read (to the host)
                e = free_slot(slot_of(k - LAG));
                gate.store(to_dev ? k - LAG + 1 + XFER_SLOTS : k - LAG + 1, std::memory_order_release);
            }
            if (k >= n || e != hipSuccess) continue;
            if (to_dev) wait_done(k);
            else if (k >= XFER_SLOTS) wait_done(k - XFER_SLOTS);
            e = launch(k);
        }
        if (e != hipSuccess) stop.store(true);
        for (auto& t : pool) t.join();
        return e;
    }

private:
    template <class S, class Lo, class Hi, class Launch, class Host>
    hipError_t serial(bool to_dev, int64_t n, S slot_of, Lo lo, Hi hi, Launch launch, Host host) {
        hipError_t e = hipSuccess;
        if (to_dev) {
            for (int64_t k = 0; k < n && e == hipSuccess; k++) {
                e = free_slot(slot_of(k));
                if (e != hipSuccess) break;
                host(lo(k), hi(k), slot(slot_of(k)));
                e = launch(k);
            }
            return e;
        }
        // to the host: kernels run up to a ring ahead of the copies
        for (int64_t k = 0, l = 0; k < n && e == hipSuccess; k++) {
            for (; l < n && l < k + XFER_SLOTS && e == hipSuccess; l++) {
                e = free_slot(slot_of(l));
                if (e == hipSuccess) e = launch(l);
            }
            if (e == hipSuccess) e = free_slot(slot_of(k));
            if (e == hipSuccess) host(lo(k), hi(k), slot(slot_of(k)));
        }
        return e;
    }
};

// The host side of a transfer of whole grids: grid g's elements
// [start[g], start[g + 1]) lie at ptr(g) in the heap.
template <class Ptr>
inline void xfer_pieces(bool to_slot, const std::vector<int64_t>& start, Ptr ptr, int64_t e0, int64_t e1,
                        double* slot) {
    size_t g = std::upper_bound(start.begin(), start.end(), e0) - start.begin() - 1;
    for (int64_t e = e0; e < e1; g++) {
        const int64_t end = std::min(e1, start[g + 1]);
        if (end <= e) continue;
        double* h = ptr(g) + (e - start[g]);
        if (to_slot) std::memcpy(slot + (e - e0), h, (end - e) * sizeof(double));
        else std::memcpy(h, slot + (e - e0), (end - e) * sizeof(double));
        e = end;
    }
}

}  // namespace amrgpu
