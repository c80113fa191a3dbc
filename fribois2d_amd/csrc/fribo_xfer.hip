// State transfer (fribo_set_state / fribo_get_state / fribo_fetch_fields and
// the named field reads) between the device fields, whose rows are padded to
// the pitch P, and the caller's contiguous arrays.
//
// A pitched copy of the runtime costs about 8 us per row whatever the row's
// length (2.6 ms for the state of a 64x48 grid, 84 ms at 2048x1536), so the
// rows are packed by a kernel that writes pinned host memory directly, all
// arrays of the call as one flat range cut into chunks of at most 4 MB.
// Where there are several, three chunks are in flight: while the kernels of
// the next two run, the host copies the finished one out.  Up to seven helper
// threads copy where there is enough to copy (first writes to fresh pages cost
// a single thread several times the PCIe time).  A transfer of one chunk runs
// its kernel, then its copy: 0.25 ms for a state of 2 MB.  The pressure's pending means are subtracted by the
// kernel.  Uploads take the same way back.  The whole state's read-back:
// 83.7 -> 5.8 ms at 2048x1536 (22 GB/s into fresh host pages), 13.6 -> 0.36
// ms at 384x288, 2.6 -> 0.04 ms at 64x48.
#include "fribo_xfer.h"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace {

struct XferTab {
    double* dev[XFER_MAXSEG];
    unsigned off[XFER_MAXSEG + 1];   // first flat element of each segment
    int n[XFER_MAXSEG], pitch[XFER_MAXSEG], k0[XFER_MAXSEG], pressure[XFER_MAXSEG];
    int nseg;
};

// Flat elements [o, o + len) of the transfer, element o + i in stage[i].
// Bound by PCIe: one 8-byte element per lane, consecutive lanes on
// consecutive elements, so a wave moves 512 contiguous bytes on both sides.
template <bool PUT>
__global__ __launch_bounds__(256) void k_xfer(const XferTab T, unsigned o, unsigned len, double* __restrict__ stage,
                                              const DevScalars* __restrict__ S, int n2, int n3m)
{
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < len; i += gridDim.x * 256) {
        const unsigned f = o + i;
        int s = 0;
        while (s + 1 < T.nseg && f >= T.off[s + 1]) ++s;
        const unsigned r = f - T.off[s], row = r / (unsigned)T.n[s], col = r - row * (unsigned)T.n[s];
        double* d = T.dev[s] + (size_t)row * T.pitch[s] + col;
        if (PUT) {
            *d = stage[i];
        } else {
            double v = *d;
            if (T.pressure[s]) {
                const int k = T.k0[s] + (int)row;
                v = v - ((k < 1 || k > n3m || (int)col == n2 - 1) ? S->goff : S->pend);
            }
            stage[i] = v;
        }
    }
}

// Host side of the flat range [a, b) of a chunk that starts at o.
void host_copy(const XferTab& T, double* const* host, unsigned o, double* stage, unsigned a, unsigned b, bool put)
{
    for (int s = 0; s < T.nseg; ++s) {
        const unsigned lo = std::max(a, T.off[s]), hi = std::min(b, T.off[s + 1]);
        if (lo >= hi) continue;
        double* h = host[s] + (lo - T.off[s]);
        double* g = stage + (lo - o);
        if (put) memcpy(g, h, (size_t)(hi - lo) * sizeof(double));
        else memcpy(h, g, (size_t)(hi - lo) * sizeof(double));
    }
}

// Helper threads of one transfer: each copies its share of every chunk that
// is posted.  A thread that cannot be started leaves its share to the others.
class Crew {
public:
    Crew(int want, const XferTab& T, double* const* host, bool put) : T_(T), host_(host), put_(put)
    {
        try {
            th_.reserve(want);
            for (int i = 0; i < want; ++i) th_.emplace_back([this, i] { work(i + 1); });
        } catch (const std::exception&) {
        }
    }
    ~Crew()
    {
        {
            std::lock_guard<std::mutex> l(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto& t : th_) t.join();
    }
    // Copies the chunk [o, o + len), with every helper.
    void run(unsigned o, unsigned len, double* stage)
    {
        const unsigned parts = (unsigned)th_.size() + 1;
        if (parts > 1) {
            std::lock_guard<std::mutex> l(mu_);
            o_ = o;
            len_ = len;
            stage_ = stage;
            left_ = parts - 1;
            ++seq_;
        }
        if (parts > 1) cv_.notify_all();
        share(0, parts, o, len, stage);
        if (parts > 1) {
            std::unique_lock<std::mutex> l(mu_);
            done_.wait(l, [this] { return left_ == 0; });
        }
    }

private:
    void share(unsigned i, unsigned parts, unsigned o, unsigned len, double* stage)
    {
        const unsigned a = (unsigned)((unsigned long long)len * i / parts);
        const unsigned b = (unsigned)((unsigned long long)len * (i + 1) / parts);
        host_copy(T_, host_, o, stage, o + a, o + b, put_);
    }
    void work(unsigned i)
    {
        unsigned seen = 0;
        for (;;) {
            unsigned o, len, parts;
            double* stage;
            {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return stop_ || seq_ != seen; });
                if (seq_ == seen) return;
                seen = seq_;
                o = o_;
                len = len_;
                stage = stage_;
                parts = (unsigned)th_.size() + 1;
            }
            share(i, parts, o, len, stage);
            {
                std::lock_guard<std::mutex> l(mu_);
                if (--left_ == 0) done_.notify_one();
            }
        }
    }
    const XferTab& T_;
    double* const* host_;
    const bool put_;
    std::vector<std::thread> th_;
    std::mutex mu_;
    std::condition_variable cv_, done_;
    unsigned seq_ = 0, o_ = 0, len_ = 0, left_ = 0;
    double* stage_ = nullptr;
    bool stop_ = false;
};

constexpr size_t kChunk = 512 * 1024;   // doubles: 4 MB
constexpr int SLOTS = XferEvents::SLOTS;

// Pinned staging blocks.  A transfer leases one and is complete when it gives
// it back, so a block serves every handle, stream and thread in turn, and
// there are as many as transfers run at once (each handle with a block of its
// own kept up to 12 MB of locked memory, 3 GB with 256 of them, and allocated
// it in its first transfer).  Sizes are powers of two of 1 MB up to the
// largest a transfer can use, 12 MB; a block that is too small is replaced.
// At most kIdle blocks wait for the next transfer.
struct Block {
    double* p = nullptr;
    size_t n = 0;      // doubles
    int dev = -1;
};
constexpr int kIdle = 8;
std::mutex g_mu;
Block g_idle[kIdle];
size_t g_held = 0;     // doubles in idle and leased blocks
int g_users = 0;

hipError_t lease(int dev, size_t want, Block& b)
{
    size_t n = 128 * 1024;
    while (n < want) n *= 2;
    n = std::min<size_t>(n, SLOTS * kChunk);
    Block old;
    {
        std::lock_guard<std::mutex> l(g_mu);
        Block *fit = nullptr, *small = nullptr;
        for (auto& q : g_idle) {
            if (!q.p || q.dev != dev) continue;
            if (q.n >= want) {
                if (!fit || q.n < fit->n) fit = &q;
            } else if (!small || q.n > small->n) {
                small = &q;
            }
        }
        if (fit) {
            b = *fit;
            *fit = Block();
            return hipSuccess;
        }
        if (small) {
            old = *small;
            *small = Block();
        }
        g_held += n;
        g_held -= old.n;
    }
    if (old.p) hipHostFree(old.p);
    b.dev = dev;
    b.n = n;
    const hipError_t e = hipHostMalloc((void**)&b.p, n * sizeof(double), hipHostMallocDefault);
    if (e != hipSuccess) {
        b = Block();
        std::lock_guard<std::mutex> l(g_mu);
        g_held -= n;
    }
    return e;
}

void give(Block& b)
{
    if (!b.p) return;
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (g_users > 0)
            for (auto& q : g_idle)
                if (!q.p) {
                    q = b;
                    return;
                }
        g_held -= b.n;
    }
    hipHostFree(b.p);
}

}  // namespace

void xfer_attach()
{
    std::lock_guard<std::mutex> l(g_mu);
    ++g_users;
}

void xfer_detach()
{
    Block out[kIdle];
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (--g_users > 0) return;
        for (int i = 0; i < kIdle; ++i) {
            out[i] = g_idle[i];
            g_idle[i] = Block();
            g_held -= out[i].n;
        }
    }
    for (auto& q : out)
        if (q.p) hipHostFree(q.p);
}

// Bytes of pinned staging memory the library holds.
extern "C" long fribo_staging_bytes(void)
{
    std::lock_guard<std::mutex> l(g_mu);
    return (long)(g_held * sizeof(double));
}

void xfer_free(XferEvents& R)
{
    for (auto& e : R.ev) {
        if (e) hipEventDestroy(e);
        e = nullptr;
    }
}

hipError_t xfer_run(XferEvents& R, int dev, const FluidDev& F, XferSeg* segs, int nseg, bool put, hipStream_t st)
{
    XferTab T{};
    double* host[XFER_MAXSEG];
    unsigned total = 0;
    for (int s = 0; s < nseg; ++s) {
        T.dev[s] = segs[s].dev;
        host[s] = segs[s].host;
        T.n[s] = segs[s].n;
        T.pitch[s] = segs[s].pitch;
        T.k0[s] = segs[s].k0;
        T.pressure[s] = segs[s].pressure;
        T.off[s] = total;
        total += (unsigned)segs[s].n * (unsigned)segs[s].rows;
    }
    T.nseg = nseg;
    T.off[nseg] = total;
    // nothing selected: still wait, and report what the stream's work ended with
    if (total == 0) return hipStreamSynchronize(st);
    hipError_t e = hipSuccess;
    const DeviceGuard guard(dev);
    for (auto& ev : R.ev)
        if (!ev && (e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return e;
    const unsigned chunk = (unsigned)std::min<size_t>(kChunk, total), nc = (total + chunk - 1) / chunk;
    Block b;
    if ((e = lease(dev, (size_t)std::min<unsigned>(SLOTS, nc) * chunk, b)) != hipSuccess) return e;
    auto slot = [&](unsigned c) { return b.p + (size_t)(c % SLOTS) * chunk; };
    auto len = [&](unsigned c) { return std::min(chunk, total - c * chunk); };
    auto wait = [&](unsigned c) { return hipEventSynchronize(R.ev[c % SLOTS]); };
    auto launch = [&](unsigned c) {
        const unsigned l = len(c);
        const dim3 g(std::min(1024u, (l + 255) / 256));
        if (put) hipLaunchKernelGGL(k_xfer<true>, g, dim3(256), 0, st, T, c * chunk, l, slot(c), F.S, F.n2, F.n3m);
        else hipLaunchKernelGGL(k_xfer<false>, g, dim3(256), 0, st, T, c * chunk, l, slot(c), F.S, F.n2, F.n3m);
        const hipError_t le = hipGetLastError();
        return le != hipSuccess ? le : hipEventRecord(R.ev[c % SLOTS], st);
    };
    const size_t bytes = (size_t)total * sizeof(double);
    const int helpers = bytes >= (size_t)16 << 20 ? 7 : bytes >= (size_t)2 << 20 ? 3 : 0;
    // the kernels of the first chunks run while the helpers start
    if (!put)
        for (unsigned c = 0; c < std::min<unsigned>(SLOTS, nc) && e == hipSuccess; ++c) e = launch(c);
    if (e == hipSuccess) {
        Crew crew(helpers, T, host, put);
        for (unsigned c = 0; c < nc && e == hipSuccess; ++c) {
            // put: the slot's last kernel has read it; get: the chunk's
            // kernel has written it
            if ((!put || c >= SLOTS) && (e = wait(c)) != hipSuccess) break;
            crew.run(c * chunk, len(c), slot(c));
            const unsigned nx = put ? c : c + SLOTS;
            if (nx < nc) e = launch(nx);
        }
        // the block is free again when the last kernels have read it
        if (put && e == hipSuccess) e = wait(nc - 1);
    }
    if (e != hipSuccess) hipStreamSynchronize(st);
    give(b);
    return e;
}
