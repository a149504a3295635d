// vah_transfer.h -- states between the padded device fields and the caller's
// interior arrays.
//
// What bounds a transfer is the host side: e, p and u of 201x201x101 cells (196 MB)
// were copied whole into a pageable buffer, its pages touched for the first time,
// then picked out of it cell by cell with two divisions per element, and took 130 of
// the 226 ms of an output interval of 40 steps (97 ms with the same kernels).  A
// checkpoint of 201x201 cells (25 fields up, 30 down) went from 6.9 to 1.34 ms.
// Here chunks of whole rows, at most kSlotBytes (or one row, where it is longer), go
// through slots that the owner keeps, pinned from kPinnedBytes on; rows are copied
// between a slot and the caller's array while the next chunk is on the link; and from
// kParallelBytes on kWorkers host threads share the chunks (one thread copies rows at
// about 10 GB/s, a fifth of the link).
#pragma once

#include <hip/hip_runtime.h>

#include <string.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "vah_host_common.h"

namespace vah_host {

// Rows of the device fields: x fastest, g ghost cells on each side in x and y, gz
// in eta, fields fs elements apart.
struct Rows {
    long nx, ny, nz, g, gz, fs;
    explicit Rows(const Layout &l) : nx(l.nx), ny(l.ny), nz(l.nz), g(2), gz(l.nz > 1 ? 2 : 0), fs(l.fs) {}
    // interior cells alone, one field after the other
    Rows(long nx_, long ny_, long nz_) : nx(nx_), ny(ny_), nz(nz_), g(0), gz(0), fs(nx_ * ny_ * nz_) {}
    long length() const { return nx + 2 * g; }
    bool compact() const { return g == 0 && gz == 0 && fs == nx * ny * nz; }
    long per_field() const { return (ny + 2 * g) * (nz + 2 * gz); }
    // first element of row r, counted over all fields; the row after a field's last
    // starts the next field, so the gap between fields belongs to the last row
    long start(long r) const { return r / per_field() * fs + r % per_field() * length(); }
    // index of the row's first interior cell among the caller's elements, -1 for a ghost row
    long interior(long r) const {
        const long f = r / per_field(), s = r % per_field(), j = s % (ny + 2 * g) - g, k = s / (ny + 2 * g) - gz;
        return j < 0 || j >= ny || k < 0 || k >= nz ? -1 : ((f * nz + k) * ny + j) * nx;
    }
    // slot image of rows [r0, r1) -> the caller's array, and back (ghosts and gaps 0)
    void out(long r0, long r1, const double *slot, double *dst) const {
        for (long r = r0; r < r1; ++r) {
            const long m = interior(r);
            if (m >= 0) memcpy(dst + m, slot + (start(r) - start(r0)) + g, sizeof(double) * nx);
        }
    }
    void in(long r0, long r1, const double *src, double *slot) const {
        for (long r = r0; r < r1; ++r) {
            const long m = interior(r), at = start(r) - start(r0), end = start(r + 1) - start(r0);
            double *row = slot + at;
            if (m < 0) {
                memset(row, 0, sizeof(double) * (end - at));
                continue;
            }
            memset(row, 0, sizeof(double) * g);
            memcpy(row + g, src + m, sizeof(double) * nx);
            memset(row + g + nx, 0, sizeof(double) * (end - at - g - nx));
        }
    }
};

// nf fields at dev, and the caller's array (one of the two by direction).
struct Segment {
    double *dev;
    int nf;
    double *dst;
    const double *src;
};

// The slots of one context or batch.  Transfers on one object from several
// threads take turns.
class Transfer {
  public:
    ~Transfer() { release(); }

    void release() {
        if (pinned_) (void)hipHostFree(slots_);
        else delete[] slots_;
        slots_ = nullptr;
        pinned_ = false;
        nslots_ = 0;
        slot_bytes_ = 0;
    }

    // Slots for transfers of up to `bytes` in rows of `row` bytes ahead of the first.
    hipError_t reserve(size_t bytes, size_t row) {
        std::lock_guard<std::mutex> hold(lock_);
        return grow(bytes, row);
    }
    hipError_t download(int device, hipStream_t stream, const Rows &R, const std::vector<Segment> &segs) {
        return guarded(device, stream, R, segs, false);
    }
    hipError_t upload(int device, hipStream_t stream, const Rows &R, const std::vector<Segment> &segs) {
        return guarded(device, stream, R, segs, true);
    }

  private:
    static constexpr size_t kSlotBytes = 1 << 20;
    // Below this a context that lives for one short event would pay more for pinned
    // slots than it saves: create, set, one step, read and close of 41x37 cells 0.88 ms
    // with them, 0.47 ms with pageable slots (0.73 ms before).  From here on they pay: a
    // checkpoint of 201x201 cells 1.45 ms, 1.95 ms pageable, when both were measured; the
    // whole life of such a context takes 1.35 ms (9.8 ms before).
    static constexpr size_t kPinnedBytes = 4 << 20;
    static constexpr size_t kParallelBytes = 16 << 20;  // below, starting threads costs what they save
    static constexpr int kWorkers = 4, kDepth = 2;      // slots per worker: one on the link, one being copied

    std::mutex lock_;
    char *slots_ = nullptr;
    bool pinned_ = false, refused_ = false;
    int nslots_ = 0;
    size_t slot_bytes_ = 0;

    hipError_t grow(size_t bytes, size_t row) {
        const int n = kDepth * (bytes >= kParallelBytes ? kWorkers : 1);
        const size_t size = std::max(row, std::min(bytes, kSlotBytes));
        const bool pin = pinned_ || bytes >= kPinnedBytes;
        if (slots_ && n <= nslots_ && size <= slot_bytes_ && (!pin || pinned_ || refused_))
            return hipSuccess;
        const int want = std::max(n, nslots_);
        const size_t each = std::max(size, slot_bytes_);
        if (pinned_) (void)hipHostFree(slots_);
        else delete[] slots_;
        nslots_ = 0;
        slot_bytes_ = 0;
        slots_ = nullptr;
        void *p = nullptr;
        pinned_ = pin && !refused_ && hipHostMalloc(&p, want * each) == hipSuccess;
        if (pin && !pinned_) {  // pageable slots work too
            refused_ = true;
            (void)hipGetLastError();
        }
        slots_ = pinned_ ? (char *)p : new (std::nothrow) char[want * each];
        if (!slots_) return hipErrorOutOfMemory;
        nslots_ = want;
        slot_bytes_ = each;
        return hipSuccess;
    }

    // no exception leaves a C entry
    hipError_t guarded(int device, hipStream_t stream, const Rows &R, const std::vector<Segment> &segs, bool up) {
        try {
            return run(device, stream, R, segs, up);
        } catch (const std::bad_alloc &) {
            return hipErrorOutOfMemory;
        }
    }

    hipError_t straight(hipStream_t stream, const Rows &R, const std::vector<Segment> &segs, bool up) {
        hipError_t e = hipSuccess;
        for (const Segment &s : segs) {
            const size_t bytes = sizeof(double) * s.nf * R.fs;
            if (e == hipSuccess)
                e = up ? hipMemcpyAsync(s.dev, s.src, bytes, hipMemcpyHostToDevice, stream)
                       : hipMemcpyAsync(s.dst, s.dev, bytes, hipMemcpyDeviceToHost, stream);
        }
        const hipError_t w = hipStreamSynchronize(stream);
        return e == hipSuccess ? w : e;
    }

    struct Chunk {
        int seg;
        long r0, r1;
    };

    hipError_t run(int device, hipStream_t stream, const Rows &R, const std::vector<Segment> &segs, bool up) {
        std::lock_guard<std::mutex> hold(lock_);
        const size_t row = sizeof(double) * (R.length() + 64);  // with the gap behind a field's last row
        size_t bytes = 0;
        for (const Segment &s : segs) bytes += sizeof(double) * s.nf * R.fs;
        if (!bytes) return hipSuccess;
        // Fields without ghosts and no pinned slots: straight between the caller's arrays
        // and the device, one wait for all (the five maps of vah_validity, 41x37 cells: 125
        // us through pageable slots, 86 so)
        if (R.compact() && !pinned_ && bytes < kPinnedBytes) return straight(stream, R, segs, up);
        hipError_t e = grow(bytes, row);
        if (e != hipSuccess) return e;
        std::vector<Chunk> chunks;
        for (int s = 0; s < (int)segs.size(); ++s) {
            const long rows = segs[s].nf * R.per_field();
            const long step = std::max(1L, (long)((slot_bytes_ - 64 * 8) / (sizeof(double) * R.length())));
            for (long r = 0; r < rows; r += step) {
                long r1 = std::min(rows, r + step);
                // the gaps between fields count too
                while (r1 > r + 1 && sizeof(double) * (R.start(r1) - R.start(r)) > slot_bytes_) --r1;
                chunks.push_back({s, r, r1});
                r = r1 - step;
            }
        }
        const int workers = bytes >= kParallelBytes ? kWorkers : 1;
        hipError_t err[kWorkers] = {};
        auto work = [&](int w) { err[w] = share(device, stream, R, segs, chunks, w, workers, up); };
        std::thread helper[kWorkers];
        for (int w = 1; w < workers; ++w) {
            try {
                helper[w] = std::thread(work, w);
            } catch (...) {  // no thread to be had: this share is done below
            }
        }
        work(0);
        for (int w = 1; w < workers; ++w) {
            if (helper[w].joinable()) helper[w].join();
            else work(w);
        }
        e = hipStreamSynchronize(stream);
        for (int w = 0; w < workers; ++w)
            if (e == hipSuccess) e = err[w];
        return e;
    }

    // Chunks w, w + workers, ... through two slots: one copy of this share is on the link
    // while the host copies the chunk before it (down) or after it (up).  Waits are for
    // the stream: with an event per chunk, waited for, the runtime took 0.7 to 2.8 ms
    // longer over the next stream, allocation and pageable copy of the process (creating
    // the next context of 201x201 cells 0.26 -> 2.6 ms), however the events were made or
    // kept; recorded but not waited for they cost nothing.
    hipError_t share(int device, hipStream_t stream, const Rows &R, const std::vector<Segment> &segs,
                     const std::vector<Chunk> &chunks, int w, int workers, bool up) {
        hipError_t e = w ? hipSetDevice(device) : hipSuccess;
        auto slot = [&](size_t n) { return (double *)(slots_ + (w * kDepth + n / workers % kDepth) * slot_bytes_); };
        auto copy = [&](size_t n) {
            const Chunk &c = chunks[n];
            double *dev = segs[c.seg].dev + R.start(c.r0);
            const size_t bytes = sizeof(double) * (R.start(c.r1) - R.start(c.r0));
            return up ? hipMemcpyAsync(dev, slot(n), bytes, hipMemcpyHostToDevice, stream)
                      : hipMemcpyAsync(slot(n), dev, bytes, hipMemcpyDeviceToHost, stream);
        };
        if (!up && e == hipSuccess && (size_t)w < chunks.size()) e = copy(w);
        for (size_t n = w; e == hipSuccess && n < chunks.size(); n += workers) {
            const Chunk &c = chunks[n];
            if (up) {
                R.in(c.r0, c.r1, segs[c.seg].src, slot(n));
                if (n >= (size_t)workers) e = hipStreamSynchronize(stream);  // the other slot is free
                if (e == hipSuccess) e = copy(n);
                continue;
            }
            e = hipStreamSynchronize(stream);
            if (e == hipSuccess && n + workers < chunks.size()) e = copy(n + workers);
            if (e == hipSuccess) R.out(c.r0, c.r1, slot(n), segs[c.seg].dst);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing in flight on the slots
        return e;
    }
};

}  // namespace vah_host
