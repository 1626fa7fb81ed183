// mpsq_buffers.h -- device buffers and job tables of the host side.  The
// includer brings the HIP runtime's declarations and the MPSQ_ERR_* codes.
#pragma once
#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <vector>

namespace mpsq {

struct Err {
    int code;
};

#define HIPCHK(x)                                                                                                     \
    do {                                                                                                              \
        hipError_t e_ = (x);                                                                                          \
        if (e_ != hipSuccess) throw Err{MPSQ_ERR_DEVICE};                                                             \
    } while (0)

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    bool lent = false;  // the memory is the caller's
    // use the caller's memory (which outlives the buffer's use of it)
    void adopt(void *q, size_t b)
    {
        release();
        p = q;
        bytes = b;
        lent = true;
    }
    void ensure(size_t b)
    {
        if (b <= bytes && p) return;
        release();
        if (b == 0) return;
        if (hipMalloc(&p, b) != hipSuccess) {
            p = nullptr;
            throw Err{MPSQ_ERR_DEVICE};
        }
        bytes = b;
    }
    void release()
    {
        if (p && !lent) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
        lent = false;
    }
    template <typename T> T *as() const { return static_cast<T *>(p); }
    ~DevBuf() { release(); }
};

// A device table made from a few numbers (its key), uploaded again when they
// change.  The key is dropped first, so that a table whose allocation fails is
// made anew by the next call and not taken for the old one.
template <typename T> struct KeyedTable {
    DevBuf d;
    std::vector<T> h;
    std::array<int64_t, 3> key{};
    bool valid = false;
    // fill: writes the n entries
    template <typename F> const T *get(const std::array<int64_t, 3> &k, size_t n, hipStream_t st, F fill)
    {
        if (!valid || key != k) {
            valid = false;
            h.assign(n, T{});
            fill(h.data());
            d.ensure(sizeof(T) * n);
            HIPCHK(hipMemcpyAsync(d.p, h.data(), sizeof(T) * n, hipMemcpyHostToDevice, st));
            key = k;
            valid = true;
        }
        return d.template as<T>();
    }
};

// ---------------------------------------------------------------------------
// Job tables: built in pinned host memory and uploaded with one copy per
// run, ahead of the kernels that read them (stream order).  Before the host
// rewrites the tables it waits for the previous upload, which keeps a
// pending copy from reading half-written tables.
// ---------------------------------------------------------------------------
struct Arena {
    unsigned char *h = nullptr;
    size_t cap = 0, used = 0;
    DevBuf d;
    hipEvent_t ev = nullptr;
    bool pending = false;
    // what the device has: the first `sent` bytes, uploaded on sent_st; tables
    // equal to it (a plan's next points, an engine's next batch of frames) are
    // not uploaded again
    size_t sent = 0;
    hipStream_t sent_st = nullptr;
    bool dirty = true;
    void begin()
    {
        used = 0;
        dirty = sent == 0;
    }
    // wait for a copy still reading the host tables
    void settle()
    {
        if (pending) HIPCHK(hipEventSynchronize(ev));
        pending = false;
    }
    // before the host tables change: they are no longer what the device has,
    // also if the tables being put are never finished (an allocation throws)
    void diverge()
    {
        settle();
        sent = 0;
        dirty = true;
    }
    size_t put_raw(const void *src, size_t bytes)
    {
        const size_t off = (used + 255) & ~(size_t)255;
        if (off + bytes > cap) {
            size_t nc = std::max<size_t>(cap * 2, 1 << 16);
            while (nc < off + bytes) nc *= 2;
            diverge();
            unsigned char *nh = nullptr;
            HIPCHK(hipHostMalloc(reinterpret_cast<void **>(&nh), nc, hipHostMallocDefault));
            if (h) {
                std::memcpy(nh, h, used);
                (void)hipHostFree(h);
            }
            h = nh;
            cap = nc;
        }
        if (bytes && (dirty || off + bytes > sent || std::memcmp(h + off, src, bytes) != 0)) {
            diverge();
            std::memcpy(h + off, src, bytes);
        }
        used = off + bytes;
        return off;
    }
    template <typename T> size_t put(const std::vector<T> &v) { return put_raw(v.data(), sizeof(T) * v.size()); }
    void upload(hipStream_t st)
    {
        if (used == 0 || (!dirty && used <= sent && st == sent_st)) return;
        sent = 0;
        d.ensure(used);
        if (!ev) HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        HIPCHK(hipMemcpyAsync(d.p, h, used, hipMemcpyHostToDevice, st));
        HIPCHK(hipEventRecord(ev, st));
        pending = true;
        sent = used;
        sent_st = st;
    }
    template <typename T> const T *dev(size_t off) const
    {
        return reinterpret_cast<const T *>(static_cast<const unsigned char *>(d.p) + off);
    }
    ~Arena()
    {
        if (pending && ev) (void)hipEventSynchronize(ev);
        if (ev) (void)hipEventDestroy(ev);
        if (h) (void)hipHostFree(h);
    }
};

}  // namespace mpsq
