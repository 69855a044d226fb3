// A result array that the caller has just allocated has no pages yet, and one thread that copies into it
// faults them in one after the other: 4 GB/s (9 GB/s with huge pages) against 57 GB/s of DMA from an
// MI355X to pinned memory; the two fields of 64 modes on 24^3 SU(3) (340 MB) took 36 ms to read back.
// Here up to MAX_WORKERS threads copy (and fault) chunks of CHUNK bytes from a ring of SLOTS pinned
// buffers, while the calling thread keeps the DMA of the next chunks in flight: about 20 GB/s.  An array
// whose pages exist goes faster without it (8.4 MB: 260 us plain, 340 us through the ring; 2100 and 710 us
// when fresh), and so does every upload (8.4 MB: 260 against 340 us).  Pinned arrays take the DMA directly
// (170 MB: 3.1 ms, 5.6 ms through the ring).
#include "ovl_hostcopy.hpp"

#include <sched.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

namespace ovl {

namespace {

constexpr size_t CHUNK = (size_t)1 << 20;
constexpr int SLOTS = 16, MAX_WORKERS = 8;

// whole CPUs of the quota in a control group's directory (version 2: cpu.max "QUOTA PERIOD", version 1: two
// files); a large number without one
int group_quota(const std::string &dir)
{
    constexpr int NONE = 1 << 20;
    double quota = -1, period = -1;
    std::ifstream max(dir + "/cpu.max");
    if (max) {
        std::string q;
        max >> q >> period;
        if (q != "max") quota = std::atof(q.c_str());
    } else {
        std::ifstream(dir + "/cpu.cfs_quota_us") >> quota;
        std::ifstream(dir + "/cpu.cfs_period_us") >> period;
    }
    if (!(quota > 0 && period > 0)) return NONE;
    return (int)std::min<double>(NONE, std::max(1.0, std::floor(quota / period)));
}

// the smallest quota of the process's control group and those above it
int quota_cpus(const std::string &root)
{
    int cpus = std::min(group_quota(root), std::min(group_quota(root + "/cpu"), group_quota(root + "/cpu,cpuacct")));
    std::ifstream self("/proc/self/cgroup");
    for (std::string line; std::getline(self, line);) {
        if (line.compare(0, 3, "0::") != 0) continue;
        for (std::string path = line.substr(3); path.size() > 1; path.resize(path.rfind('/')))
            cpus = std::min(cpus, group_quota(root + path));
    }
    return cpus;
}

// More spinning threads than the process may run at once would be stopped by the scheduler in the middle of a
// copy, so a container's quota counts as much as the affinity mask.
int cpus_allowed(const char *cgroup_root)
{
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof set, &set) != 0) return 1;
    return std::min(CPU_COUNT(&set), quota_cpus(cgroup_root ? cgroup_root : "/sys/fs/cgroup"));
}

// whether the HIP runtime knows the memory (pinned, managed or device memory): the DMA reaches it without a
// copy by the host, and mincore says nothing about its pages (a driver mapping has none in the page cache)
bool known_to_hip(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

// whether the array's pages are mostly not there yet (a sample of them)
bool untouched(const void *p, size_t bytes)
{
    const size_t page = (size_t)sysconf(_SC_PAGESIZE);
    constexpr int SAMPLES = 16;
    int absent = 0;
    for (int k = 0; k < SAMPLES; ++k) {
        const size_t at = ((size_t)p + bytes / SAMPLES * k + bytes / (2 * SAMPLES)) / page * page;
        unsigned char there = 1;
        if (mincore((void *)at, page, &there) != 0) return false;
        absent += !(there & 1);
    }
    return absent > SAMPLES / 2;
}

// one copy: chunk i is [i CHUNK, min(bytes, (i + 1) CHUNK)) and uses slot i % SLOTS
struct Job {
    char *host = nullptr;
    size_t bytes = 0;
    long n = 0;
    std::atomic<long> next{0};     // next chunk a worker takes
    std::atomic<long> limit{0};    // chunks below it have arrived in their slots
    std::atomic<bool> stop{false};
    std::vector<std::atomic<char>> done;
    explicit Job(long chunks) : n(chunks), done((size_t)chunks)
    {
        for (auto &d : done) d.store(0, std::memory_order_relaxed);
    }
    size_t len(long i) const { return std::min(CHUNK, bytes - (size_t)i * CHUNK); }
};

// waits are a few microseconds (a DMA or a copy of one chunk): spin, giving the core away now and then
template <class F> void spin_until(F ready)
{
    for (int k = 0; !ready(); ++k)
        if (k % 64 == 63) std::this_thread::yield();
}

class Ring {
public:
    // null when the process has no second core, or no pinned memory or threads are to be had
    static Ring *make()
    {
        const int nw = std::min(MAX_WORKERS, cpus_allowed(nullptr) - 1);
        if (nw < 1) return nullptr;
        std::unique_ptr<Ring> r(new Ring);
        r->events_.reserve(SLOTS);
        r->threads_.reserve((size_t)nw);
        bool ok = hipHostMalloc((void **)&r->pinned_, CHUNK * SLOTS, hipHostMallocDefault) == hipSuccess;
        if (!ok) (void)hipGetLastError();
        for (int k = 0; ok && k < SLOTS; ++k) {
            hipEvent_t e = nullptr;
            ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
            if (ok) r->events_.push_back(e);
        }
        ok = ok && hipGetDevice(&r->device_) == hipSuccess;
        if (ok) {
            try {
                for (int k = 0; k < nw; ++k) r->threads_.emplace_back([p = r.get()] { p->worker(); });
            } catch (...) {  // std::system_error: no more threads
                ok = !r->threads_.empty();
            }
        }
        return ok ? r.release() : nullptr;
    }

    ~Ring()
    {
        {
            std::lock_guard<std::mutex> l(mu_);
            quit_ = true;
        }
        cv_.notify_all();
        for (auto &t : threads_) t.join();
        for (auto e : events_) (void)hipEventDestroy(e);
        if (pinned_) (void)hipHostFree(pinned_);
    }

    int device() const { return device_; }

    hipError_t to_host(char *host, const char *dev, size_t bytes, hipStream_t st)
    {
        Job j((long)((bytes + CHUNK - 1) / CHUNK));
        j.host = host;
        j.bytes = bytes;
        start(&j);
        hipError_t e = hipSuccess;
        long issued = 0;
        for (long i = 0; i < j.n && e == hipSuccess; ++i) {
            // keep the DMA ahead as far as emptied slots allow; chunk i itself must have one
            for (; issued < j.n && issued < i + SLOTS && e == hipSuccess; ++issued) {
                if (issued >= SLOTS && !finished(j, issued - SLOTS)) {
                    if (issued > i) break;
                    spin_until([&] { return finished(j, issued - SLOTS); });
                }
                e = hipMemcpyAsync(slot(issued), dev + (size_t)issued * CHUNK, j.len(issued), hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(events_[(size_t)(issued % SLOTS)], st);
            }
            if (e == hipSuccess) e = wait(events_[(size_t)(i % SLOTS)]);
            if (e == hipSuccess) j.limit.store(i + 1, std::memory_order_release);
        }
        return finish(&j, e, st);
    }

private:
    // a chunk's DMA takes 20 us: polled, since a blocking wait costs as much again to wake
    static hipError_t wait(hipEvent_t ev)
    {
        hipError_t e;
        spin_until([&] { return (e = hipEventQuery(ev)) != hipErrorNotReady; });
        return e;
    }

    char *slot(long i) const { return pinned_ + (size_t)(i % SLOTS) * CHUNK; }
    static bool finished(const Job &j, long i) { return j.done[(size_t)i].load(std::memory_order_acquire) != 0; }

    void start(Job *j)
    {
        {
            std::lock_guard<std::mutex> l(mu_);
            job_ = j;
            ++serial_;
            busy_ = (int)threads_.size();
        }
        cv_.notify_all();
    }

    // waits for the workers to leave the job and for the stream; the slots are free afterwards
    hipError_t finish(Job *j, hipError_t e, hipStream_t st)
    {
        if (e != hipSuccess) j->stop.store(true, std::memory_order_release);
        {
            std::unique_lock<std::mutex> l(mu_);
            idle_.wait(l, [this] { return busy_ == 0; });
            job_ = nullptr;
        }
        const hipError_t s = hipStreamSynchronize(st);
        return e != hipSuccess ? e : s;
    }

    void run(Job *j)
    {
        for (;;) {
            const long i = j->next.fetch_add(1, std::memory_order_relaxed);
            if (i >= j->n) return;
            spin_until([&] {
                return j->limit.load(std::memory_order_acquire) > i || j->stop.load(std::memory_order_acquire);
            });
            if (j->stop.load(std::memory_order_acquire)) return;
            std::memcpy(j->host + (size_t)i * CHUNK, slot(i), j->len(i));
            j->done[(size_t)i].store(1, std::memory_order_release);
        }
    }

    void worker()
    {
        long seen = 0;
        for (;;) {
            Job *j;
            {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return quit_ || serial_ != seen; });
                if (quit_) return;
                seen = serial_;
                j = job_;
            }
            run(j);
            {
                std::lock_guard<std::mutex> l(mu_);
                if (--busy_ == 0) idle_.notify_all();
            }
        }
    }

    char *pinned_ = nullptr;
    int device_ = 0;
    std::vector<hipEvent_t> events_;
    std::vector<std::thread> threads_;
    std::mutex mu_;
    std::condition_variable cv_, idle_;
    Job *job_ = nullptr;
    long serial_ = 0;
    int busy_ = 0;
    bool quit_ = false;
};

std::mutex g_mu;  // the ring, its holders and its use: one copy at a time
Ring *g_ring = nullptr;
bool g_tried = false;
int g_holders = 0;
std::atomic<long> g_copies{0};  // copies that took the ring

// the ring, locked for one copy of this thread on the current device; null: copy plainly
Ring *take_ring(std::unique_lock<std::mutex> &lock)
{
    lock = std::unique_lock<std::mutex>(g_mu, std::try_to_lock);
    if (!lock.owns_lock() || g_holders == 0) return nullptr;
    if (!g_ring && !g_tried) {
        g_tried = true;
        g_ring = Ring::make();
    }
    int dev = -1;
    if (!g_ring || hipGetDevice(&dev) != hipSuccess || dev != g_ring->device()) return nullptr;
    return g_ring;
}

}  // namespace

hipError_t copy_to_host(void *host, const void *dev, size_t bytes, hipStream_t st)
{
    if (bytes >= HOSTCOPY_MIN && untouched(host, bytes) && !known_to_hip(host)) {
        std::unique_lock<std::mutex> lock;
        try {
            if (Ring *r = take_ring(lock)) {
                g_copies.fetch_add(1, std::memory_order_relaxed);
                return r->to_host((char *)host, (const char *)dev, bytes, st);
            }
        } catch (const std::bad_alloc &) {  // of the ring or of the job, before any thread has the job
        }
    }
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
}

void hostcopy_hold()
{
    std::lock_guard<std::mutex> l(g_mu);
    ++g_holders;
}

void hostcopy_release()
{
    std::lock_guard<std::mutex> l(g_mu);
    if (--g_holders > 0) return;
    delete g_ring;
    g_ring = nullptr;
    g_tried = false;
}

}  // namespace ovl

extern "C" long ovl_hostcopy_ring_copies() { return ovl::g_copies.load(std::memory_order_relaxed); }

extern "C" int ovl_hostcopy_cpus(const char *cgroup_root) { return ovl::cpus_allowed(cgroup_root); }
