// Products into the caller's host arrays.
//
// The device holds maps as four doubles per pixel and the inverse pixel
// matrices as six; the caller gets [npix][nmap] and [npix][nmap][nmap].  A
// kernel lays each piece out and writes it straight into pinned host memory,
// and a few threads carry the pieces on into the caller's (pageable, often
// untouched) arrays, so that the transfer, the page faults and the copies of
// different pieces run at the same time.  The runtime's own pageable copy
// moves under a megabyte at a time through one bounce buffer on one thread,
// and the layouts were then turned on the host: the maps and baselines of 16
// detectors x 2^24 samples at Nside 512 (685 MB) took 145 ms that way and take
// 15 ms (45 GB/s) now, those of 4 x 2^22 at Nside 256 (123 MB) 30 and 3.4 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <vector>

#include "madam_context.hpp"
#include "madam_workers.hpp"

namespace madam {

// ------------------------------------------------------------------ layout kernel

static constexpr int OUT_TPB = 256;
static constexpr int OUT_MAX_PIECES = 12;

struct OutPiece {
    int kind;
    const void *src;
    int64_t e0, n;     // output elements e0 .. e0 + n - 1
    void *out;         // where element e0 goes
};
struct OutPieces {
    OutPiece p[OUT_MAX_PIECES];
};

__global__ void __launch_bounds__(OUT_TPB) k_out_pack(OutPieces ps)
{
    const OutPiece p = ps.p[blockIdx.y];
    const int sym[9] = {0, 1, 2, 1, 3, 4, 2, 4, 5};
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < p.n; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t t = p.e0 + i;
        if (p.kind == OUT_COPY4) {
            ((int32_t *)p.out)[i] = ((const int32_t *)p.src)[t];
            continue;
        }
        const double *src = (const double *)p.src;
        double v;
        switch (p.kind) {
        case OUT_MAP3: v = src[t / 3 * 4 + t % 3]; break;
        case OUT_MAP1: v = src[t * 4]; break;
        case OUT_CC9: {
            int a = (int)(t % 9), b = 0;
#pragma unroll
            for (int k = 0; k < 9; ++k) b = a == k ? sym[k] : b;
            v = src[t / 9 * 6 + b];
            break;
        }
        case OUT_CC1: v = src[t * 6]; break;
        default: v = src[t]; break;
        }
        ((double *)p.out)[i] = v;
    }
}

static size_t elem_bytes(int kind) { return kind == OUT_COPY4 ? 4 : 8; }

static void launch_out(hipStream_t s, const OutPieces &ps, int np)
{
    int64_t most = 1;
    for (int i = 0; i < np; ++i) most = std::max(most, ps.p[i].n);
    unsigned g = (unsigned)std::min<int64_t>((most + OUT_TPB - 1) / OUT_TPB, 1024);
    k_out_pack<<<dim3(g, (unsigned)np), OUT_TPB, 0, s>>>(ps);
    MADAM_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------ pinned slots
// At most OUT_SLOTS slots of OUT_SLOT bytes for all handles of the process,
// lent to one call at a time and freed when the last handle goes.

static constexpr size_t OUT_SLOT = 4 << 20;
static constexpr int OUT_SLOTS = 8;
static std::mutex g_out_mu;
static std::vector<void *> g_out_free;
static int g_out_made = 0, g_out_handles = 0;

void out_handle_made()
{
    std::lock_guard<std::mutex> lk(g_out_mu);
    ++g_out_handles;
}

void out_handle_gone()
{
    std::lock_guard<std::mutex> lk(g_out_mu);
    if (--g_out_handles > 0) return;
    for (void *p : g_out_free) (void)hipHostFree(p);
    g_out_made -= (int)g_out_free.size();
    g_out_free.clear();
}

// a slot, or null when all are lent (or memory is short)
static void *slot_take()
{
    std::lock_guard<std::mutex> lk(g_out_mu);
    if (!g_out_free.empty()) {
        void *p = g_out_free.back();
        g_out_free.pop_back();
        return p;
    }
    if (g_out_made >= OUT_SLOTS) return nullptr;
    g_out_free.reserve(OUT_SLOTS);   // giving a slot back cannot fail
    void *p = nullptr;
    if (hipHostMalloc(&p, OUT_SLOT, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    ++g_out_made;
    return p;
}

// up to `want` slots, given back once the kernels on the stream that write them have ended
struct SlotLease {
    std::vector<void *> p;
    hipStream_t s;
    SlotLease(int want, hipStream_t st) : s(st)
    {
        p.reserve(want);
        while ((int)p.size() < want) {
            void *q = slot_take();
            if (!q) break;
            p.push_back(q);
        }
    }
    ~SlotLease()
    {
        if (p.empty()) return;
        (void)hipStreamSynchronize(s);
        std::lock_guard<std::mutex> lk(g_out_mu);
        for (void *q : p) g_out_free.push_back(q);
    }
};

// ------------------------------------------------------------------ copies

static constexpr size_t OUT_SMALL = 1 << 20;   // one launch and one copy up to here

void copy_out(Context &c, const std::vector<OutItem> &items)
{
    hipStream_t s = c.stream;
    // an error that an earlier call of the caller's left is not one of the launches below
    (void)hipGetLastError();
    size_t total = 0;
    for (const OutItem &it : items) total += (size_t)it.n * elem_bytes(it.kind) + 8;
    DBuf<char> d;
    if (total <= OUT_SMALL && if_room([&] { d.alloc(total); })) {
        // everything in one launch into device scratch, and one copy
        std::vector<char> h(total);
        OutPieces ps;
        size_t off = 0, i0 = 0;
        std::vector<size_t> at;
        for (size_t i = 0; i < items.size(); ++i) {
            at.push_back(off);
            ps.p[i - i0] = OutPiece{items[i].kind, items[i].src, 0, items[i].n, d.p + off};
            off += ((size_t)items[i].n * elem_bytes(items[i].kind) + 7) / 8 * 8;
            if (i + 1 - i0 == OUT_MAX_PIECES || i + 1 == items.size()) {
                launch_out(s, ps, (int)(i + 1 - i0));
                i0 = i + 1;
            }
        }
        d2h(h.data(), d.p, off, s);
        MADAM_CHECK(hipStreamSynchronize(s));
        for (size_t i = 0; i < items.size(); ++i)
            memcpy(items[i].dst, h.data() + at[i], (size_t)items[i].n * elem_bytes(items[i].kind));
        return;
    }
    struct Chunk {
        int item;
        int64_t e0, n;
    };
    std::vector<Chunk> chunks;
    for (size_t i = 0; i < items.size(); ++i) {
        int64_t per = (int64_t)(OUT_SLOT / elem_bytes(items[i].kind));
        for (int64_t e = 0; e < items[i].n; e += per) chunks.push_back({(int)i, e, std::min(per, items[i].n - e)});
    }
    std::atomic<size_t> next{0};
    std::mutex mu;
    hipError_t err = hipSuccess;
    auto work = [&](void *slot) {
        hipEvent_t ev = nullptr;
        hipError_t e = hipSetDevice(c.device);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        while (e == hipSuccess) {
            size_t k = next++;
            if (k >= chunks.size()) break;
            const OutItem &it = items[chunks[k].item];
            {
                std::lock_guard<std::mutex> lk(mu);
                if (err != hipSuccess) break;
                OutPieces ps;
                ps.p[0] = OutPiece{it.kind, it.src, chunks[k].e0, chunks[k].n, slot};
                unsigned g = (unsigned)std::min<int64_t>((chunks[k].n + OUT_TPB - 1) / OUT_TPB, 1024);
                k_out_pack<<<dim3(g, 1), OUT_TPB, 0, s>>>(ps);
                e = hipGetLastError();
                if (e == hipSuccess) e = hipEventRecord(ev, s);
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev);
            size_t eb = elem_bytes(it.kind);
            if (e == hipSuccess) memcpy((char *)it.dst + chunks[k].e0 * eb, slot, (size_t)chunks[k].n * eb);
        }
        if (ev) (void)hipEventDestroy(ev);
        if (e != hipSuccess) {
            std::lock_guard<std::mutex> lk(mu);
            if (err == hipSuccess) err = e;
        }
    };
    // a thread per 8 MB: 685 MB take 63 / 34 / 20 / 15 ms with 1 / 2 / 4 / 8
    // threads, 36 MB 2.0 / 1.3 / 1.0 / 1.1
    int want = (int)std::min<size_t>((total + 2 * OUT_SLOT - 1) / (2 * OUT_SLOT), OUT_SLOTS);
    SlotLease slots(want, s);
    if (slots.p.empty()) {
        // every slot is lent: lay out in device scratch and let the runtime copy
        with_room(c, [&] { d.alloc(OUT_SLOT); });
        for (const Chunk &ck : chunks) {
            const OutItem &it = items[ck.item];
            size_t eb = elem_bytes(it.kind);
            OutPieces ps;
            ps.p[0] = OutPiece{it.kind, it.src, ck.e0, ck.n, d.p};
            launch_out(s, ps, 1);
            d2h((char *)it.dst + ck.e0 * eb, d.p, (size_t)ck.n * eb, s);
        }
        MADAM_CHECK(hipStreamSynchronize(s));
        return;
    }
    run_workers((int)slots.p.size(), [&](int i) { work(slots.p[i]); });
    MADAM_CHECK(err);
    MADAM_CHECK(hipStreamSynchronize(s));
}

}  // namespace madam
