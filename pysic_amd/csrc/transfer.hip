// transfer.hip -- per-atom arrays and scalars between host and device.
//
// The C-ABI speaks in the caller's atom order and in rows of 3 doubles; the
// device holds cell-sorted double4.  The kernels here translate while they
// read or write pinned host memory directly, so a transfer is one pass over
// the bus (24 bytes an atom instead of 32, no copy through a device staging
// array, no pageable copy).  The order is translated on the device side of
// the bus, through the inverse permutation, so the host side is contiguous.
//
// Pinned memory: every system holds one block (the mail words and two small
// slots, alternated so that an upload need not wait for the one before it);
// longer arrays go through 3 MiB slots, two for each of up to PAIRS copying
// threads, in chunks, one slot filled while the other is emptied (one thread
// cannot keep up with the bus: the caller's pages are often touched for the
// first time here).  Pinning costs more than most transfers, so blocks and
// slots are kept for the next user, a bounded number of each, and are freed
// with the last system.
//
// Scalars (energies, virials, flags, hashes) are written by the kernels that
// form them, or by k_report, straight into the pinned `mail` words: a call
// that needs them on the host waits for the stream once and reads them.
//
// Measured: 50 MD steps of 1,048,576 atoms and their positions and momenta in
// fresh numpy arrays 39.5 -> 21.2 ms (the steps are 18.8 of them); two
// evaluations (coordinates in, lists, energy, forces out) of 4,096 atoms 0.70
// -> 0.34 ms, where each made ten device-side copies of 4 us and waited nine
// times and now waits three times; forces of 561,934 atoms out 1.9 -> 0.5 ms.
#include "system.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

namespace {

constexpr size_t SMALL = 256 << 10;          // bytes of a block's two slots, each
constexpr size_t BLOCK = 1024 + 2 * SMALL;   // mail words first
constexpr size_t SLOT = 3 << 20;
constexpr size_t KEEP_BLOCKS = 16, KEEP_SLOTS = 2 * HostLink::PAIRS;
static_assert(MAIL_WORDS * sizeof(double) <= 1024, "the mail fits its part of the block");

// What is kept, for all systems and threads of the process.  Pinned portably:
// any device may use it next.  Coherent by its own flag, whatever the process
// sets as the default: the host reads rows and error words after an event,
// which need not flush a device's caches to memory of the other kind.
struct Pinned {
    std::mutex m;
    long users = 0;
    std::vector<char *> block, slot;

    static char *fresh(size_t bytes)
    {
        char *p = nullptr;
        HIP_TRY(hipHostMalloc((void **)&p, bytes, hipHostMallocPortable | hipHostMallocCoherent));
        return p;
    }
    char *take(std::vector<char *> &v, size_t bytes)
    {
        {
            std::lock_guard<std::mutex> g(m);
            if (!v.empty()) {
                char *p = v.back();
                v.pop_back();
                return p;
            }
        }
        return fresh(bytes);
    }
    void give(std::vector<char *> &v, size_t keep, char *p)
    {
        {
            std::lock_guard<std::mutex> g(m);
            if (users > 0 && v.size() < keep) {
                v.push_back(p);
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void enter()
    {
        std::lock_guard<std::mutex> g(m);
        ++users;
    }
    void leave()
    {
        std::lock_guard<std::mutex> g(m);
        if (--users > 0) return;
        for (char *p : block) (void)hipHostFree(p);
        for (char *p : slot) (void)hipHostFree(p);
        block.clear();
        slot.clear();
    }
};
Pinned &pinned()
{
    static Pinned *p = new Pinned;   // outlives every static destructor
    return *p;
}

constexpr int TB = 256;

__global__ void k_invert(int n, const int *__restrict__ id, int *__restrict__ inv)
{
    const int s = blockIdx.x * TB + threadIdx.x;
    if (s < n) inv[id[s]] = s;
}

// rows [first, first + rows) of the caller's order, x, y, z of double4 src;
// a thread per double, so the bus sees whole lines
__global__ void k_pack3(int rows, const int *__restrict__ inv, const double4 *__restrict__ src,
                        double *__restrict__ out)
{
    const int t = blockIdx.x * TB + threadIdx.x, r = t / 3;
    if (r < rows) out[t] = ((const double *)(src + inv[r]))[t - 3 * r];
}
__global__ void k_unpack3(int rows, const int *__restrict__ inv, const double *__restrict__ in,
                          double4 *__restrict__ dst)
{
    const int t = blockIdx.x * TB + threadIdx.x, r = t / 3;
    if (r < rows) ((double *)(dst + inv[r]))[t - 3 * r] = in[t];
}
__global__ void k_pack1(int rows, const int *__restrict__ inv, const double *__restrict__ src,
                        double *__restrict__ out)
{
    const int r = blockIdx.x * TB + threadIdx.x;
    if (r < rows) out[r] = src[inv ? inv[r] : r];
}
__global__ void k_unpack1(int rows, const int *__restrict__ inv, const double *__restrict__ in,
                          double *__restrict__ dst)
{
    const int r = blockIdx.x * TB + threadIdx.x;
    if (r < rows) dst[inv[r]] = in[r];
}

__global__ void k_report(const double *__restrict__ t, const double *__restrict__ g,
                         const int *__restrict__ flags, double *__restrict__ mail)
{
    const int i = threadIdx.x;
    if (i < 7) mail[i] = t ? t[i] : 0.0;
    else if (i < 14) mail[i] = g ? g[i - 7] : 0.0;
    else if (i < 18) ((int *)(mail + 14))[i - 14] = flags[i - 14];
}

char *block(System &S)
{
    HostLink &L = S.link;
    if (!L.block) {
        pinned().enter();
        try {
            L.block = pinned().take(pinned().block, BLOCK);
        } catch (...) {
            pinned().leave();
            throw;
        }
    }
    return L.block;
}

hipEvent_t event(System &S, int k)
{
    hipEvent_t &e = S.link.done[k];
    if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return e;
}

// The next small slot, once the upload that used it last has read it.
char *small_slot(System &S)
{
    HostLink &L = S.link;
    char *base = block(S);
    const int k = L.turn ^= 1;
    if (L.busy[k]) {
        HIP_TRY(hipEventSynchronize(event(S, k)));
        L.busy[k] = false;
    }
    return base + 1024 + k * SMALL;
}

// body(thread) on as many threads as there are chunks, up to the slot pairs;
// the first failure is thrown here, after all have ended
template <class Body>
void on_threads(System &S, int chunks, Body &&body)
{
    const int T = chunks < HostLink::PAIRS ? chunks : HostLink::PAIRS;
    (void)block(S);   // counts this system among the slots' users
    PysicError err[HostLink::PAIRS];
    bool bad[HostLink::PAIRS] = {};
    auto guarded = [&](int t) {
        char *pair[2] = {nullptr, nullptr};
        try {
            HIP_TRY(hipSetDevice(S.device));
            for (char *&p : pair) p = pinned().take(pinned().slot, SLOT);
            body(t, T, pair);
        } catch (const PysicError &e) {
            err[t] = e;
            bad[t] = true;
        } catch (const std::exception &e) {
            err[t] = PysicError{PYSIC_ENOMEM, e.what()};
            bad[t] = true;
        }
        // a failed body may have left a kernel on the slots
        if (bad[t]) (void)hipStreamSynchronize(S.stream);
        for (char *p : pair)
            if (p) pinned().give(pinned().slot, KEEP_SLOTS, p);
    };
    std::thread helper[HostLink::PAIRS];
    int started = 1;
    try {
        for (; started < T; ++started) helper[started] = std::thread(guarded, started);
    } catch (const std::exception &) {
        // no more threads: their chunks are done below
    }
    guarded(0);
    for (int t = started; t < T; ++t) guarded(t);
    for (int t = 1; t < started; ++t) helper[t].join();
    for (int t = 0; t < T; ++t)
        if (bad[t]) throw err[t];
}

// `rows` rows of `width` doubles to the host; pack(first, count, out) launches
// the kernel that writes rows [first, first + count) into out.  `ready` is
// asked after the stream has been waited for; without its consent the host
// array stays as it is.
template <class Pack>
void to_host(System &S, int rows, int width, double *host, Pack &&pack,
             const std::function<bool()> &ready = nullptr)
{
    const size_t row = sizeof(double) * width;
    if (row * rows <= SMALL) {
        char *p = small_slot(S);
        pack(0, rows, (double *)p);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(S.stream));
        if (!ready || ready()) std::memcpy(host, p, row * rows);
        return;
    }
    if (ready) {
        HIP_TRY(hipStreamSynchronize(S.stream));
        if (!ready()) return;
    }
    const int per = (int)(SLOT / row), chunks = (rows + per - 1) / per;
    on_threads(S, chunks, [&](int t, int T, char **pair) {
        int held = -1;   // the chunk in flight
        auto take = [&](int c) {
            const int k = (c / T) % 2, first = c * per;
            HIP_TRY(hipEventSynchronize(event(S, 2 * t + k)));
            std::memcpy((char *)host + row * first, pair[k], row * std::min(per, rows - first));
        };
        for (int c = t; c < chunks; c += T) {
            const int k = (c / T) % 2, first = c * per;
            pack(first, std::min(per, rows - first), (double *)pair[k]);
            HIP_TRY(hipGetLastError());
            HIP_TRY(hipEventRecord(event(S, 2 * t + k), S.stream));
            if (held >= 0) take(held);
            held = c;
        }
        if (held >= 0) take(held);
    });
}

// the other way; returns with the caller's array read and, where it went
// through the small slots, the kernel queued on the stream
template <class Unpack>
void from_host(System &S, int rows, int width, const double *host, Unpack &&unpack)
{
    const size_t row = sizeof(double) * width;
    if (row * rows <= SMALL) {
        char *p = small_slot(S);
        const int k = S.link.turn;
        std::memcpy(p, host, row * rows);
        unpack(0, rows, (const double *)p);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(event(S, k), S.stream));
        S.link.busy[k] = true;
        return;
    }
    const int per = (int)(SLOT / row), chunks = (rows + per - 1) / per;
    on_threads(S, chunks, [&](int t, int T, char **pair) {
        bool used[2] = {false, false};
        for (int c = t; c < chunks; c += T) {
            const int k = (c / T) % 2, first = c * per, count = std::min(per, rows - first);
            if (used[k]) HIP_TRY(hipEventSynchronize(event(S, 2 * t + k)));
            std::memcpy(pair[k], (const char *)host + row * first, row * count);
            unpack(first, count, (const double *)pair[k]);
            HIP_TRY(hipGetLastError());
            HIP_TRY(hipEventRecord(event(S, 2 * t + k), S.stream));
            used[k] = true;
        }
        for (int k = 0; k < 2; ++k)
            if (used[k]) HIP_TRY(hipEventSynchronize(event(S, 2 * t + k)));
    });
}

const int *inverse(System &S)
{
    S.inv.ensure(S.n);
    k_invert<<<div_up(S.n, TB), TB, 0, S.stream>>>(S.n, S.id.p, S.inv.p);
    HIP_TRY(hipGetLastError());
    return S.inv.p;
}

}  // namespace

double *sys_mail(System &S) { return (double *)block(S); }

void sys_post_report(System &S, bool tersoff, bool general)
{
    k_report<<<1, 64, 0, S.stream>>>(tersoff ? S.totals.p : nullptr,
                                     general ? S.gtotals.p : nullptr, S.flags.p, sys_mail(S));
    HIP_TRY(hipGetLastError());
}

Report sys_read_report(System &S)
{
    Report r;
    std::memcpy(r.t, sys_mail(S), sizeof(r.t));
    std::memcpy(r.g, sys_mail(S) + 7, sizeof(r.g));
    std::memcpy(r.f, sys_mail(S) + 14, sizeof(r.f));
    return r;
}

void sys_download3(System &S, const double4 *src, double *host, const std::function<bool()> &ready)
{
    const int *inv = inverse(S);
    to_host(S, S.n, 3, host, [&](int first, int count, double *out) {
        k_pack3<<<div_up(3 * count, TB), TB, 0, S.stream>>>(count, inv + first, src, out);
    }, ready);
}

void sys_download1(System &S, const double *src, double *host)
{
    const int *inv = inverse(S);
    to_host(S, S.n, 1, host, [&](int first, int count, double *out) {
        k_pack1<<<div_up(count, TB), TB, 0, S.stream>>>(count, inv + first, src, out);
    });
}

void sys_download_plain(System &S, int count, const double *src, double *host)
{
    to_host(S, count, 1, host, [&](int first, int rows, double *out) {
        k_pack1<<<div_up(rows, TB), TB, 0, S.stream>>>(rows, nullptr, src + first, out);
    });
}

void sys_upload3(System &S, const double *host, double4 *dst)
{
    const int *inv = inverse(S);
    from_host(S, S.n, 3, host, [&](int first, int count, const double *in) {
        k_unpack3<<<div_up(3 * count, TB), TB, 0, S.stream>>>(count, inv + first, in, dst);
    });
}

void sys_upload1(System &S, const double *host, double *dst)
{
    const int *inv = inverse(S);
    from_host(S, S.n, 1, host, [&](int first, int count, const double *in) {
        k_unpack1<<<div_up(count, TB), TB, 0, S.stream>>>(count, inv + first, in, dst);
    });
}

void HostLink::release()
{
    for (hipEvent_t &e : done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    busy[0] = busy[1] = false;
    if (!block) return;
    pinned().give(pinned().block, KEEP_BLOCKS, block);
    block = nullptr;
    pinned().leave();
}
