// State transfer (fribo_set_state / fribo_get_state / fribo_fetch_fields and
// the named field reads) between the device fields, whose rows are padded to
// the pitch P, and the caller's contiguous arrays.
//
// A pitched copy of the runtime costs about 8 us per row whatever the row's
// length (2.6 ms for the state of a 64x48 grid, 84 ms at 2048x1536), so the
// rows are packed by a kernel that writes pinned host memory directly, all
// arrays of the call as one flat range cut into chunks of at most 4 MB.
// Three chunks are in flight: while the kernels of the next two run, the host
// copies the finished one out, with up to seven helper threads where there is
// enough to copy (first writes to fresh pages cost a single thread several
// times the PCIe time).  The pressure's pending means are subtracted by the
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

}  // namespace

void xfer_free(XferRing& R)
{
    if (R.stage) hipHostFree(R.stage);
    R.stage = nullptr;
    R.chunk = 0;
    for (auto& e : R.ev) {
        if (e) hipEventDestroy(e);
        e = nullptr;
    }
}

hipError_t xfer_run(XferRing& R, const FluidDev& F, XferSeg* segs, int nseg, bool put, hipStream_t st)
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
    if (total == 0) return hipSuccess;
    hipError_t e = hipSuccess;
    for (auto& ev : R.ev)
        if (!ev && (e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return e;
    const size_t want = std::min<size_t>(kChunk, total);
    if (R.chunk < want) {
        // a put of an earlier call may still read the ring
        if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
        if (R.stage) hipHostFree(R.stage);
        R.stage = nullptr;
        R.chunk = 0;
        e = hipHostMalloc((void**)&R.stage, want * XferRing::SLOTS * sizeof(double), hipHostMallocDefault);
        if (e != hipSuccess) return e;
        R.chunk = want;
    }
    constexpr int NS = XferRing::SLOTS;
    const unsigned chunk = (unsigned)R.chunk, nc = (total + chunk - 1) / chunk;
    auto slot = [&](unsigned c) { return R.stage + (size_t)(c % NS) * chunk; };
    auto len = [&](unsigned c) { return std::min(chunk, total - c * chunk); };
    auto launch = [&](unsigned c) {
        const unsigned l = len(c);
        const dim3 g(std::min(1024u, (l + 255) / 256));
        if (put) hipLaunchKernelGGL(k_xfer<true>, g, dim3(256), 0, st, T, c * chunk, l, slot(c), F.S, F.n2, F.n3m);
        else hipLaunchKernelGGL(k_xfer<false>, g, dim3(256), 0, st, T, c * chunk, l, slot(c), F.S, F.n2, F.n3m);
        const hipError_t le = hipGetLastError();
        return le != hipSuccess ? le : hipEventRecord(R.ev[c % NS], st);
    };
    const size_t bytes = (size_t)total * sizeof(double);
    const int helpers = bytes >= (size_t)16 << 20 ? 7 : bytes >= (size_t)2 << 20 ? 3 : 0;
    // the kernels of the first chunks run while the helpers start
    if (!put)
        for (unsigned c = 0; c < std::min<unsigned>(NS, nc); ++c)
            if ((e = launch(c)) != hipSuccess) return e;
    Crew crew(helpers, T, host, put);
    for (unsigned c = 0; c < nc; ++c) {
        // put: the slot's last kernel (of this call or an earlier one) has read it;
        // get: the chunk's kernel has written it
        if ((e = hipEventSynchronize(R.ev[c % NS])) != hipSuccess) return e;
        crew.run(c * chunk, len(c), slot(c));
        const unsigned nx = put ? c : c + NS;
        if (nx < nc && (e = launch(nx)) != hipSuccess) return e;
    }
    return hipSuccess;
}
