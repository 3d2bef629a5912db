// persist.cpp -- admission of kernels whose workgroups wait for each other
// (persist.hpp).
#include "persist.hpp"

#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>

namespace self {

namespace {

struct Flight {
    int device;
    hipStream_t stream;
    double demand, share;  // CUs' worth of workgroups; a workgroup's share of a CU
    hipEvent_t done;
    unsigned long long group;
};

// Launches of one group may run side by side; each waits for the groups before.
unsigned long long g_group = 1;

std::mutex g_mutex;
std::vector<Flight> g_flights;
std::vector<std::pair<int, hipEvent_t>> g_events;  // finished flights' events, by device

void prune()
{
    size_t k = 0;
    for (Flight &f : g_flights) {
        if (hipEventQuery(f.done) == hipErrorNotReady) g_flights[k++] = f;
        else g_events.emplace_back(f.device, f.done);
    }
    g_flights.resize(k);
    (void)hipGetLastError();  // "not ready" is an answer here, not an error of a later call
}

}  // namespace

int persist_cus(int device)
{
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    return n;
}

int persist_blocks_per_cu(const void *kernel, int threads)
{
    static std::mutex m;
    static std::map<std::pair<const void *, int>, int> known;
    std::lock_guard<std::mutex> lock(m);
    auto it = known.find({kernel, threads});
    if (it != known.end()) return it->second;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess) {
        (void)hipGetLastError();
        n = 0;
    }
    known[{kernel, threads}] = n;
    return n;
}

// Half a microsecond to one a poll.  SELF_AMD_SPIN_LIMIT overrides it (a test of
// the fallback sets 0: the first unsuccessful poll gives up).
unsigned persist_spin_limit()
{
    const char *s = std::getenv("SELF_AMD_SPIN_LIMIT");
    if (s && *s) return (unsigned)std::strtoul(s, nullptr, 10);
    return 2000;
}

int ResidentRuns::clear(hipStream_t s)
{
    SELF_HIP(hipMemsetAsync(messages, 0, messageBytes, s));
    SELF_HIP(hipMemsetAsync(status, 0, sizeof(int), s));
    *hostStatus = 0;
    tag = 0;
    return SELF_OK;
}

hipError_t ResidentRuns::alloc_host()
{
    if (hostStatus) return hipSuccess;
    const hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&hostStatus), sizeof(int), hipHostMallocDefault);
    if (e != hipSuccess) hostStatus = nullptr;
    return e;
}

void ResidentRuns::free_host()
{
    if (hostStatus) (void)hipHostFree(hostStatus);
    hostStatus = nullptr;
}

int ResidentRuns::settle(hipStream_t s, std::vector<Run> &again)
{
    again.clear();
    if (pending.empty()) return SELF_OK;
    SELF_HIP(hipStreamSynchronize(s));
    const int bad = *static_cast<volatile int *>(hostStatus);
    std::vector<Run> done;
    done.swap(pending);
    if (bad == 0) {
        ups.finished();
        return SELF_OK;
    }
    ups.gaveUp();
    if (int rc = clear(s)) return rc;
    size_t first = 0;
    while (first < done.size() && done[first].launch != bad) ++first;
    SELF_REQUIRE(first < done.size(), SELF_ERR_HIP, "a resident launch gave up and cannot be found (%d)", bad);
    again.assign(done.begin() + (long)first, done.end());
    return SELF_OK;
}

// Alone on the device, `blocks` <= perCu x CUs workgroups of one kernel all
// become resident.  Beside others, by shares of a CU: a workgroup of share s
// finds no room only if every CU has more than 1 - s in use, that is, if the
// launches in flight use more than CUs x (1 - s) together; half the device is
// kept free beyond that, since the room on a CU need not be in one piece.
// Where every launch takes a CU a workgroup, each needs only as many CUs as it
// has.  Launches on one stream run one after another and count once.
PersistGate::PersistGate(int device, hipStream_t stream, int blocks, int perCu)
    : rc(SELF_OK), lock_(g_mutex), device_(device), stream_(stream), demand_((double)blocks / perCu), share_(1.0 / perCu)
{
    // room for this launch's records: nothing may throw once it is queued
    g_flights.reserve(g_flights.size() + 1);
    g_events.reserve(g_events.size() + g_flights.size() + 1);
    prune();
    std::map<hipStream_t, double> per;
    double largest = share_;
    bool wholeCu = perCu == 1;
    for (const Flight &f : g_flights) {
        if (f.device != device || f.stream == stream || f.group != g_group) continue;
        double &d = per[f.stream];
        if (f.demand > d) d = f.demand;
        if (f.share > largest) largest = f.share;
        wholeCu = wholeCu && f.share == 1.0;
    }
    double sum = demand_;
    for (const auto &p : per) sum += p.second;
    const int cus = persist_cus(device);
    const bool fits = per.empty() || (wholeCu ? sum <= cus : sum <= 0.5 * cus * (1.0 - largest));
    if (!fits) ++g_group;
    for (const Flight &f : g_flights) {
        if (f.device != device || f.stream == stream || f.group == g_group) continue;
        const hipError_t e = hipStreamWaitEvent(stream, f.done, 0);
        if (e != hipSuccess && rc == SELF_OK) rc = hip_fail(e, "hipStreamWaitEvent", __FILE__, __LINE__);
    }
}

int PersistGate::launched()
{
    hipEvent_t ev = nullptr;
    for (size_t k = 0; k < g_events.size(); ++k)
        if (g_events[k].first == device_) {
            ev = g_events[k].second;
            g_events.erase(g_events.begin() + (long)k);
            break;
        }
    hipError_t e = ev ? hipSuccess : hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(ev, stream_);
    if (e != hipSuccess) {  // without its event the launch cannot be waited for by others: wait here
        (void)hipStreamSynchronize(stream_);
        if (ev) g_events.emplace_back(device_, ev);
        return hip_fail(e, "persistent launch event", __FILE__, __LINE__);
    }
    g_flights.push_back({device_, stream_, demand_, share_, ev, g_group});
    return SELF_OK;
}

}  // namespace self
