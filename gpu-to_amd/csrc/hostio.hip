// Host arrays of an entry point to and from the device.
//
// A copy of pageable memory runs on the calling thread through the runtime's
// own staging, the caller waits for it, and the checks and sign changes of an
// entry point are further passes of one thread over the array: at 192x96x96
// (43.6 MB vectors) a solve spent 1.5 ms per upload of F, 1.5 ms looking for
// NaN, 2.4 ms on the download of U and 1.0 ms on its signs, and reading a
// design's state into new arrays took 8 ms, most of it page faults.  Here the
// array goes in chunks through pinned slots of the handle: a few threads copy
// (and check) their chunks while the device moves the earlier ones: 1.2 ms up
// with the check, 1.2 ms down, 2.5 ms for the design's state.
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

#include "gputo_internal.h"

namespace gputo {

namespace {

// Four threads copy at the rate of the link (two do 40 GB/s, eight no more
// than four).  A chunk of 2 MB keeps the fixed cost of a transfer (8 us) at a
// fifth of its time; small arrays are cut into eight so that the copies and
// the transfers still overlap, down to 512 KB.  A second thread is worth its
// start (20 us) from a few MB on.
constexpr int kThreads = 4;
constexpr size_t kSlotBytes = 2 << 20, kMinChunk = 512 << 10, kBytesPerThread = 4 << 20;

struct Chunk {
    const HostJob *job;
    size_t off, len;
};

// exponent of all ones (infinity, NaN) carries into the sign bit
bool finite_words(const char *p, size_t bytes)
{
    unsigned long long acc = 0;
    for (size_t o = 0; o + 8 <= bytes; o += 8) {
        unsigned long long b;
        std::memcpy(&b, p + o, 8);
        acc |= (b & 0x7ff0000000000000ull) + 0x0010000000000000ull;
    }
    return !(acc >> 63);
}

}  // namespace

struct HostStage {
    int slots = 0;
    char *mem[2 * kThreads] = {};
    hipEvent_t ev[2 * kThreads] = {};
    bool busy[2 * kThreads] = {};  // a transfer from or to the slot was enqueued and not waited for
};

void stage_destroy(gputo_handle *h)
{
    if (!h->stage) return;
    for (int q = 0; q < h->stage->slots; ++q) {
        (void)hipHostFree(h->stage->mem[q]);
        (void)hipEventDestroy(h->stage->ev[q]);
    }
    delete h->stage;
    h->stage = nullptr;
}

static void need_slots(gputo_handle *h, int n)
{
    if (!h->stage) h->stage = new HostStage();
    HostStage &st = *h->stage;
    while (st.slots < n) {
        char *p = nullptr;
        hipEvent_t e = nullptr;
        check_hip(hipHostMalloc((void **)&p, kSlotBytes, hipHostMallocDefault), "hipHostMalloc");
        const hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        if (rc != hipSuccess) (void)hipHostFree(p);
        check_hip(rc, "hipEventCreate");
        st.mem[st.slots] = p;
        st.ev[st.slots++] = e;
    }
}

// One thread's share: the next chunk not yet taken, through two slots in turn.
// A download returns with its slots copied out; an upload's last transfers are
// left to the stream, and the slot's next user waits for them.  Errors are
// returned, not thrown.
static hipError_t worker(gputo_handle *h, bool down, const std::vector<Chunk> &chunks, std::atomic<size_t> &next,
                         std::atomic<bool> &bad, int t)
{
    HostStage &st = *h->stage;
    const Chunk *out[2] = {};  // download: what the slot holds
    hipError_t err = hipSuccess;
    auto settle = [&](int q) {
        if (st.busy[2 * t + q]) {
            const hipError_t e = hipEventSynchronize(st.ev[2 * t + q]);
            if (err == hipSuccess) err = e;
            if (out[q] && e == hipSuccess)
                std::memcpy((char *)out[q]->job->host + out[q]->off, st.mem[2 * t + q], out[q]->len);
        }
        st.busy[2 * t + q] = false;
        out[q] = nullptr;
    };
    for (int q = 0; err == hipSuccess && !bad.load(std::memory_order_relaxed);) {
        const size_t c = next.fetch_add(1);
        if (c >= chunks.size()) break;
        const Chunk &ch = chunks[c];
        const char *host = (const char *)ch.job->host + ch.off;
        if (!down && !ch.job->dev) {  // checked only
            if (!finite_words(host, ch.len)) bad = true;
            continue;
        }
        settle(q);
        if (err != hipSuccess) break;
        char *mem = st.mem[2 * t + q], *dev = (char *)ch.job->dev + ch.off;
        if (down) {
            err = hipMemcpyAsync(mem, dev, ch.len, hipMemcpyDeviceToHost, h->stream);
        } else {
            constexpr size_t kBlock = 64 << 10;  // checked while it is in a near cache
            for (size_t o = 0; o < ch.len; o += kBlock) {
                const size_t m = ch.len - o < kBlock ? ch.len - o : kBlock;
                std::memcpy(mem + o, host + o, m);
                if (ch.job->check && !finite_words(mem + o, m)) bad = true;
            }
            err = hipMemcpyAsync(dev, mem, ch.len, hipMemcpyHostToDevice, h->stream);
        }
        if (err != hipSuccess) break;
        st.busy[2 * t + q] = true;
        err = hipEventRecord(st.ev[2 * t + q], h->stream);
        out[q] = down && err == hipSuccess ? &ch : nullptr;
        q ^= 1;
        if (down) settle(q);  // copied out while the device fills the slot just given to it
    }
    if (down) {
        settle(0);
        settle(1);
    }
    return err;
}

static bool host_copy(gputo_handle *h, bool down, const HostJob *jobs, int njobs)
{
    size_t total = 0;
    for (int j = 0; j < njobs; ++j) total += jobs[j].bytes;
    size_t len = total / 8 / 8 * 8;
    if (len < kMinChunk) len = kMinChunk;
    if (len > kSlotBytes) len = kSlotBytes;
    std::vector<Chunk> chunks;
    for (int j = 0; j < njobs; ++j)
        for (size_t o = 0; o < jobs[j].bytes; o += len)
            chunks.push_back({&jobs[j], o, jobs[j].bytes - o < len ? jobs[j].bytes - o : len});
    size_t nt = 1 + total / kBytesPerThread;
    if (nt > (size_t)kThreads) nt = kThreads;
    need_slots(h, 2 * (int)nt);
    std::atomic<size_t> next{0};
    std::atomic<bool> bad{false};
    hipError_t err[kThreads] = {};
    std::vector<std::thread> th;
    th.reserve(nt);
    for (size_t t = 1; t < nt; ++t) {
        try {
            th.emplace_back([&, t] {
                err[t] = hipSetDevice(h->device);
                if (err[t] == hipSuccess) err[t] = worker(h, down, chunks, next, bad, (int)t);
            });
        } catch (...) {
            break;  // no more threads to be had: the others take all chunks
        }
    }
    err[0] = worker(h, down, chunks, next, bad, 0);
    for (std::thread &x : th) x.join();
    for (hipError_t e : err) check_hip(e, down ? "download" : "upload");
    return !bad;
}

bool host_upload(gputo_handle *h, const HostJob *jobs, int njobs) { return host_copy(h, false, jobs, njobs); }

void host_download(gputo_handle *h, const HostJob *jobs, int njobs) { host_copy(h, true, jobs, njobs); }

// u -> -u on the y components: the MATLAB frame (mgcg1.cu:282-283)
__global__ __launch_bounds__(256) void k_flip_y(double *u, long nnod)
{
    const long n = (long)blockIdx.x * 256 + threadIdx.x;
    if (n < nnod) u[3 * n + 1] = -u[3 * n + 1];
}

void launch_flip_y(hipStream_t s, double *u, long nnod)
{
    k_flip_y<<<(unsigned)((nnod + 255) / 256), 256, 0, s>>>(u, nnod);
}

}  // namespace gputo
