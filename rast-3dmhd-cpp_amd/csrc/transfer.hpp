// Fields between the host's arrays ([nz][ny][nx], ghosts included) and the
// device layout ([nz][nPy][pitch]).
//
// The planes of all fields form one sequence, moved in chunks of whole planes
// through a ring of pinned staging slabs that hold them in the host's layout:
// a device kernel packs a chunk straight into its slab (or unpacks it from
// there), adding or dropping the x, y ghosts, while the host copies other
// slabs to or from the caller's arrays with plain contiguous copies.  The
// copies of a chunk are cut into pieces that the calling thread and a few
// helpers, started once for the call, take in turn; a helper that starts late
// finds less to do and is never waited for before it has begun.
//
// The kernels read and write the pinned memory in place, at 52-53 of the
// link's 57 GB/s.  Slabs of 8 MB and more went by the copy engine through two
// device slabs before: its rate differs from machine to machine and from copy
// to copy (512x512x256 get_state 78 ms at best, 146 at worst, and 97 for
// set_state, against 83 and 83 in place whatever the machine), its set-up
// slowed first transfers, and the device slabs came on top of a server's
// budget.
//
// ms for get_state into kept arrays / set_state, FP64 (MI355X), a slab of rows
// repacked by up to 16 threads started for it -> the copy engine -> now: hydro
// 32^3 (1.6 MB) 2.3 / 2.3 -> 0.08 / 0.10 -> 0.08 / 0.11; MHD 64^3 (18 MB) 8.0 /
// 7.7 -> 0.49 / 0.56 -> 0.49 / 0.57; 128^3 (141 MB) 9.0 / 8.8 -> 5.6 / 3.1 -> 3.1
// / 3.2; 256x256x128 (554 MB) 18.7 / 14 -> 18.8 / 14 -> 11.1 / 10.9; 512x512x256
// (4.4 GB) 146 / 84 -> 146 / 97 -> 83 / 83.  The first set_state of a context:
// 128^3 9.3 -> 9.3 -> 8.4, 256x256x128 17.5 -> 20.7 -> 15.6, 512x512x256 104 -> 105
// -> 89.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "kernels_basic.hpp"

namespace mhd {

// One thread per double of a chunk's host layout: planes p0 .. p0 + np - 1 of
// the sequence (plane p: field p / nz, z = p % nz), nx = nPx + 2, ny = nPy + 2.
// periodic: the x, y ghosts take the periodic copies (3dmhdmpi.h:65-68,118-121,
// 135-142); otherwise the ghosts and the z ghost planes are zero (fluxes).
// Bound by the host link; consecutive lanes write consecutive doubles.
MHD_TU_LOCAL __global__ void __launch_bounds__(256) pack_planes_kernel(Geom g, const double* __restrict__ U, int p0,
                                                                  int np, int periodic, double* __restrict__ out)
{
    const int nx = g.nPx + 2, ny = g.nPy + 2;
    const int64_t plane = (int64_t)nx * ny, n = plane * np;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int k = (int)(i / plane);
        const int r = (int)(i - k * plane);
        int y = r / nx, x = r - y * nx;
        const int f = (p0 + k) / g.nz, z = (p0 + k) - f * g.nz;
        double v = 0.0;
        if (periodic || (x > 0 && x < nx - 1 && y > 0 && y < ny - 1 && z > 0 && z < g.nz - 1)) {
            x = x == 0 ? g.nPx - 1 : (x == nx - 1 ? 0 : x - 1);
            y = y == 0 ? g.nPy - 1 : (y == ny - 1 ? 0 : y - 1);
            v = U[f * g.fs + z * g.plane + (int64_t)y * g.pitch + x];
        }
        out[i] = v;
    }
}

// One thread per point of a chunk's device planes (pitch padding zeroed), into
// U and, when given, the second register V, whose z ghost planes no kernel
// writes.
MHD_TU_LOCAL __global__ void __launch_bounds__(256) unpack_planes_kernel(Geom g, const double* __restrict__ in, int p0,
                                                                    int np, double* __restrict__ U,
                                                                    double* __restrict__ V)
{
    const int nx = g.nPx + 2;
    const int64_t hplane = (int64_t)nx * (g.nPy + 2), n = g.plane * np;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int k = (int)(i / g.plane);
        const int r = (int)(i - k * g.plane);
        const int y = r / g.pitch, x = r - y * g.pitch;
        const int f = (p0 + k) / g.nz, z = (p0 + k) - f * g.nz;
        const double v = x < g.nPx ? in[k * hplane + (int64_t)(y + 1) * nx + x + 1] : 0.0;
        const int64_t o = f * g.fs + z * g.plane + r;
        U[o] = v;
        if (V) V[o] = v;
    }
}

// Slabs of at most 24 MB: a context pins no more than 96 MB (unless one plane
// is larger), and the first transfer has less memory to touch.  ms of the first
// set_state / a fetch into fresh arrays at 512x512x256: slabs of 64 MB 95 /
// 83.3, 32 MB 90 / 84.6, 24 MB 88 / 83.4, 16 MB 88 / 90, 8 MB 87 / 92 (too few
// huge pages in flight for the helpers).
constexpr int kSlabs = 4;
constexpr size_t kSlabBytes = 24u << 20;
constexpr size_t kPieceBytes = 256u << 10; // the smallest host copy
constexpr size_t kHugePage = 2u << 20;
constexpr size_t kCallBytes = 64u << 10;
constexpr size_t kHelperBytes = 2u << 20;  // a helper thread for each so many bytes

// The slabs and what goes with them: a domain's own, or one that the members
// of an ensemble or the runs of a server take in turn.  Nothing is allocated
// before the first transfer.
struct Staging {
    std::mutex mu;              // held for the length of a transfer
    double* host = nullptr;     // pinned, kSlabs slabs
    double* dev = nullptr;      // its device address
    size_t slab_bytes = 0;      // allocated for each
    hipEvent_t ev[kSlabs] = {}; // last kernel on each slab
};

// Planes of a slab in the transfers of nf fields of g: a quarter of the
// state, within the slab limit.
inline int staging_planes(const Geom& g, int nf)
{
    const size_t plane = (size_t)(g.nPx + 2) * (g.nPy + 2) * sizeof(double);
    const size_t total = (size_t)nf * g.nz;
    const size_t most = kSlabBytes / plane;
    const size_t n = std::min((total + kSlabs - 1) / kSlabs, most ? most : 1);
    return (int)n;
}

// Room for slabs of `want` bytes; no transfer is under way.
inline hipError_t staging_reserve(Staging& s, size_t want)
{
    hipError_t e = hipSuccess;
    for (int k = 0; k < kSlabs && e == hipSuccess; ++k)
        if (!s.ev[k]) e = hipEventCreateWithFlags(&s.ev[k], hipEventDisableTiming);
    if (e != hipSuccess || s.slab_bytes >= want) return e;
    if (s.host) (void)hipHostFree(s.host);
    s.host = s.dev = nullptr;
    s.slab_bytes = 0;
    e = hipHostMalloc(&s.host, kSlabs * want);
    if (e != hipSuccess) s.host = nullptr;
    else e = hipHostGetDevicePointer((void**)&s.dev, s.host, 0);
    if (e == hipSuccess) s.slab_bytes = want;
    return e;
}

inline void staging_destroy(Staging& s)
{
    for (hipEvent_t ev : s.ev)
        if (ev) (void)hipEventDestroy(ev);
    if (s.host) (void)hipHostFree(s.host);
}

// Copies of numbered jobs, cut into pieces that the caller and the helpers
// take in turn.  open(j) lets everyone work on job j; finish(j) works on it
// until its last piece is copied.  Jobs are opened in order; the destructor
// (also on an error return) lets the helpers go without opening the rest.
class CopyTeam {
public:
    // job j: bytes[j] bytes; copy(j, begin, end) copies a part of it; heads[j]:
    // bytes before the first huge-page boundary of its part of the caller's array
    template <typename F>
    CopyTeam(const std::vector<size_t>& bytes, const std::vector<size_t>& heads, int helpers, F copy)
        : jobs_(bytes.size())
    {
        for (size_t j = 0; j < bytes.size(); ++j) {
            Job& w = jobs_[j];
            w.bytes = bytes[j];
            // a large job in pieces of whole huge pages of the caller's array,
            // so that no two threads first touch (and zero) the same page
            const bool large = bytes[j] >= 8 * kHugePage;
            w.piece = large ? kHugePage : kPieceBytes;
            w.head = large ? heads[j] : 0;
            w.pieces = (w.bytes - w.head + w.piece - 1) / w.piece;
        }
        work_ = [this, copy](size_t j) {
            Job& w = jobs_[j];
            for (;;) {
                const size_t k = w.next.fetch_add(1, std::memory_order_relaxed);
                if (k >= w.pieces) return;
                copy(j, k ? w.head + k * w.piece : 0, std::min(w.bytes, w.head + (k + 1) * w.piece));
                w.done.fetch_add(1, std::memory_order_release);
            }
        };
        try {
            for (int t = 0; t < helpers; ++t) threads_.emplace_back([this] { helper(); });
        } catch (...) {
            // fewer helpers than asked: the caller takes their pieces
        }
    }
    ~CopyTeam()
    {
        {
            std::lock_guard<std::mutex> l(mu_);
            quit_.store(true, std::memory_order_release);
        }
        cv_.notify_all();
        for (std::thread& t : threads_) t.join();
    }
    CopyTeam(const CopyTeam&) = delete;
    CopyTeam& operator=(const CopyTeam&) = delete;

    void open(size_t j)
    {
        if (threads_.empty()) return;
        {
            std::lock_guard<std::mutex> l(mu_);
            jobs_[j].ready.store(true, std::memory_order_release);
        }
        cv_.notify_all();
    }
    void finish(size_t j)
    {
        work_(j);
        while (jobs_[j].done.load(std::memory_order_acquire) < jobs_[j].pieces) std::this_thread::yield();
    }

private:
    struct Job {
        size_t bytes = 0, piece = 0, head = 0, pieces = 0;
        std::atomic<bool> ready{false};
        std::atomic<size_t> next{0}, done{0};
    };
    void helper()
    {
        for (size_t j = 0; j < jobs_.size(); ++j) {
            auto go = [&] {
                return jobs_[j].ready.load(std::memory_order_acquire) || quit_.load(std::memory_order_acquire);
            };
            for (int k = 0; k < 64 && !go(); ++k) std::this_thread::yield();
            if (!go()) {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, go);
            }
            if (!jobs_[j].ready.load(std::memory_order_acquire)) return;
            work_(j);
        }
    }
    std::vector<Job> jobs_;
    std::function<void(size_t)> work_;
    std::mutex mu_;
    std::condition_variable cv_;
    std::atomic<bool> quit_{false};
    std::vector<std::thread> threads_;
};

// The chunks of a transfer: planes [begin, end) of the sequence.
struct ChunkPlan {
    int64_t plane;             // doubles of one host plane
    int total, per;
    int n;
    size_t slab() const { return (size_t)per * plane * sizeof(double); }
    int begin(int c) const { return c * per; }
    int planes(int c) const { return std::min(total, (c + 1) * per) - c * per; }
};

inline ChunkPlan chunk_plan(const Geom& g, int nf)
{
    ChunkPlan p;
    p.plane = (int64_t)(g.nPx + 2) * (g.nPy + 2);
    p.total = nf * g.nz;
    p.per = staging_planes(g, nf);
    p.n = (p.total + p.per - 1) / p.per;
    return p;
}

// Helper threads of a transfer of `bytes`: one for each kHelperBytes, at most
// 15 (the CPU share of one GPU on a shared host).
inline int transfer_helpers(size_t bytes)
{
    const unsigned hw = std::thread::hardware_concurrency();
    const size_t most = hw ? std::min<size_t>(hw, 16u) - 1 : 3;
    return (int)std::min(most, bytes / kHelperBytes);
}

// Calls fn(host pointer, chunk offset in bytes, length) for the parts of bytes
// [b, e) of chunk c, each within one field.
template <typename P, typename F>
inline void chunk_parts(const ChunkPlan& p, const Geom& g, P const* fields, int c, size_t b, size_t e, F fn)
{
    const size_t fbytes = (size_t)g.nz * p.plane * sizeof(double);   // one field
    size_t at = (size_t)p.begin(c) * p.plane * sizeof(double) + b;
    const size_t end = at + (e - b);
    size_t off = b;
    while (at < end) {
        const size_t f = at / fbytes, o = at - f * fbytes;
        const size_t len = std::min(end - at, fbytes - o);
        fn(fields[f], o, off, len);
        at += len;
        off += len;
    }
}

// Bytes and heads (CopyTeam) of every chunk.
template <typename P>
inline void chunk_sizes(const ChunkPlan& p, const Geom& g, P const* fields, std::vector<size_t>& bytes,
                        std::vector<size_t>& heads)
{
    bytes.resize(p.n);
    heads.resize(p.n);
    for (int c = 0; c < p.n; ++c) {
        bytes[c] = (size_t)p.planes(c) * p.plane * sizeof(double);
        const int f = p.begin(c) / g.nz, z = p.begin(c) - f * g.nz;
        const uintptr_t at = reinterpret_cast<uintptr_t>(fields[f] + z * p.plane);
        heads[c] = std::min<size_t>(bytes[c], (kHugePage - at % kHugePage) % kHugePage);
    }
}

inline int transfer_grid(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 2048); }

// The host's fields into register U (and V).  The stream orders the kernels;
// the caller holds the staging until the stream has drained.
inline hipError_t upload_fields(const Geom& g, int nf, Staging& s, hipStream_t stream, const double* const* src,
                                double* U, double* V)
try {
    const ChunkPlan p = chunk_plan(g, nf);
    hipError_t e = staging_reserve(s, p.slab());
    if (e != hipSuccess) return e;
    std::vector<size_t> bytes, heads;
    chunk_sizes(p, g, src, bytes, heads);
    auto slab = [&](double* base, int c) { return base + (size_t)(c % kSlabs) * p.per * p.plane; };
    CopyTeam team(bytes, heads, transfer_helpers((size_t)p.total * p.plane * sizeof(double)),
                  [&](size_t c, size_t b, size_t e) {
                      char* to = reinterpret_cast<char*>(slab(s.host, (int)c));
                      chunk_parts(p, g, src, (int)c, b, e, [&](const double* f, size_t o, size_t off, size_t len) {
                          std::memcpy(to + off, reinterpret_cast<const char*>(f) + o, len);
                      });
                  });
    for (int c = 0; c < p.n; ++c) {
        if (c >= kSlabs) {
            e = hipEventSynchronize(s.ev[c % kSlabs]);   // the slab's last chunk is on the device
            if (e != hipSuccess) return e;
        }
        team.open(c);
        team.finish(c);
        unpack_planes_kernel<<<transfer_grid(g.plane * p.planes(c)), 256, 0, stream>>>(g, slab(s.dev, c), p.begin(c),
                                                                                       p.planes(c), U, V);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(s.ev[c % kSlabs], stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
} catch (const std::exception&) {   // the plan's few host allocations
    return hipErrorOutOfMemory;
}

// nf fields of register U into the host arrays dst.
inline hipError_t download_fields(const Geom& g, int nf, Staging& s, hipStream_t stream, const double* U,
                                  bool periodic, double* const* dst)
try {
    const ChunkPlan p = chunk_plan(g, nf);
    hipError_t e = staging_reserve(s, p.slab());
    if (e != hipSuccess) return e;
    std::vector<size_t> bytes, heads;
    chunk_sizes(p, g, dst, bytes, heads);
    auto slab = [&](double* base, int c) { return base + (size_t)(c % kSlabs) * p.per * p.plane; };
    auto issue = [&](int c) -> hipError_t {
        pack_planes_kernel<<<transfer_grid(p.plane * p.planes(c)), 256, 0, stream>>>(g, U, p.begin(c), p.planes(c),
                                                                                     periodic ? 1 : 0, slab(s.dev, c));
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? e : hipEventRecord(s.ev[c % kSlabs], stream);
    };
    for (int c = 0; c < std::min(p.n, kSlabs); ++c) {
        e = issue(c);
        if (e != hipSuccess) return e;
    }
    CopyTeam team(bytes, heads, transfer_helpers((size_t)p.total * p.plane * sizeof(double)),
                  [&](size_t c, size_t b, size_t e) {
                      const char* from = reinterpret_cast<const char*>(slab(s.host, (int)c));
                      chunk_parts(p, g, dst, (int)c, b, e, [&](double* f, size_t o, size_t off, size_t len) {
                          // in calls short of the C library's non-temporal copies:
                          // those write around the cache lines the kernel has just
                          // zeroed in a fresh array (4.4 GB into fresh arrays: 87 ms,
                          // 83.5 so)
                          for (size_t q = 0; q < len; q += kCallBytes)
                              std::memcpy(reinterpret_cast<char*>(f) + o + q, from + off + q,
                                          std::min(kCallBytes, len - q));
                      });
                  });
    int opened = 0;
    for (int c = 0; c < p.n; ++c) {
        e = hipSuccess;
        if (opened == c) {
            e = hipEventSynchronize(s.ev[c % kSlabs]);
            if (e != hipSuccess) return e;
            team.open(opened++);
        }
        // chunks that have arrived already are open before this one is
        // finished, so that no helper waits for its last pieces
        while (opened < std::min(p.n, c + kSlabs) && (e = hipEventQuery(s.ev[opened % kSlabs])) == hipSuccess)
            team.open(opened++);
        if (e == hipErrorNotReady) (void)hipGetLastError();   // no error: later checks must not see it
        else if (e != hipSuccess) return e;
        team.finish(c);
        if (c + kSlabs < p.n) {
            e = issue(c + kSlabs);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
} catch (const std::exception&) {
    return hipErrorOutOfMemory;
}

}  // namespace mhd
