// persist.hpp -- kernels whose workgroups stay resident and wait for each
// other (several RK stages or solver iterations per launch).
//
// Exchange: up to three doubles travel as four 8-byte words (two 16-byte
// accesses), each word 48 bits of payload under the 16-bit tag of the step it
// belongs to.  A reader polls the words themselves until all carry the tag it
// wants, so no fence, flag or ordering between words is needed: an aligned
// 8-byte half of an access is single-copy atomic, and agent-scope accesses
// (sc1) are coherent across the 8 XCDs' L2s.  Flags inside the data are the
// method of the low-latency (LL) protocol of NCCL and RCCL; the words' layout,
// their tags and the bounded waits are this library's.  Buffers are double-buffered by
// the tag's parity: a writer overwrites a word only after it has received a
// value its reader sent after reading that word, so a word holds the wanted
// tag or that of two steps before and 16 bits of tag are enough.
// What bounds it is the number of accesses in flight past the L2s: with
// 32-bit tags, six 8-byte accesses a message and every lane polling until the
// slowest of its wavefront was done, 262 144 messages a stage took 91 us; with
// each lane polling for itself 18 us.
//
// Progress: a workgroup waits only for workgroups of its own launch, so every
// wait ends once all of them are resident.  PersistGate orders the process's
// own launches so that their workgroups fit beside each other, but whether the
// last workgroup is placed is not the host's to say: kernels of other streams
// that run at the start can leave a CU's LDS and registers in pieces too small
// for it (seen: a launch of 1024 workgroups beside another model's stage
// kernels).  So every wait is bounded: past `limit` polls (2000, one to two
// milliseconds, hundreds of times the longest wait of a resident launch) the launch records
// its number in *status, every other wait sees that and all workgroups end,
// leaving the launch's input untouched; the launches queued behind it return at
// once, and the host runs the steps through ordinary launches.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "common.hpp"

namespace self {

typedef unsigned long long ll_word;
typedef unsigned ll_quad __attribute__((ext_vector_type(4)));

// A message buffer: [slot][2][lane] quads, 16-byte half h of message m of a
// slot of n messages at quad (slot 2 + h) n + m.
struct LLBuf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ LLBuf(void *p, size_t bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000))
    {
    }
};

constexpr int kLLAgent = 16;                   // sc1: agent scope
constexpr int kLLPoll = 16 | (int)0x80000000;  // and volatile: each poll loads again

// bytes 0, 1 of lo16 under bytes 0, 1 of hi16
__device__ __forceinline__ unsigned ll_pair(unsigned hi16, unsigned lo16)
{
    return __builtin_amdgcn_perm(hi16, lo16, 0x05040100u);
}

// words of a message: three payloads of 48 bits, their three top halves in a fourth
__device__ __forceinline__ void ll_store3(const LLBuf &B, unsigned off0, unsigned off1, const double v[3], unsigned tag)
{
    unsigned lo[3], hi[3];
    #pragma unroll
    for (int f = 0; f < 3; ++f) {
        const ll_word b = (ll_word)__double_as_longlong(v[f]);
        lo[f] = (unsigned)b;
        hi[f] = (unsigned)(b >> 32);
    }
    const ll_quad a = {lo[0], ll_pair(tag, hi[0]), lo[1], ll_pair(tag, hi[1])};
    const ll_quad c = {lo[2], ll_pair(tag, hi[2]), (hi[0] >> 16) | (hi[1] & 0xffff0000u), (hi[2] >> 16) | (tag << 16)};
    __builtin_amdgcn_raw_buffer_store_b128(a, B.r, (int)off0, 0, kLLAgent);
    __builtin_amdgcn_raw_buffer_store_b128(c, B.r, (int)off1, 0, kLLAgent);
}

// true when every word of the message carries the tag
__device__ __forceinline__ bool ll_try3(const LLBuf &B, unsigned off0, unsigned off1, unsigned tag, double v[3])
{
    const ll_quad a = __builtin_amdgcn_raw_buffer_load_b128(B.r, (int)off0, 0, kLLPoll);
    const ll_quad c = __builtin_amdgcn_raw_buffer_load_b128(B.r, (int)off1, 0, kLLPoll);
    const unsigned T = tag << 16;
    const unsigned hi[3] = {ll_pair(c.z, a.y), (a.w & 0xffffu) | (c.z & 0xffff0000u), ll_pair(c.w, c.y)};
    const unsigned lo[3] = {a.x, a.z, c.x};
    #pragma unroll
    for (int f = 0; f < 3; ++f) v[f] = __longlong_as_double((long long)(((ll_word)hi[f] << 32) | lo[f]));
    return (((a.y ^ T) | (a.w ^ T) | (c.y ^ T) | (c.w ^ T)) >> 16) == 0;
}

// one double in one quad
__device__ __forceinline__ void ll_store1(const LLBuf &B, unsigned off, double v, unsigned tag)
{
    const ll_word b = (ll_word)__double_as_longlong(v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    const ll_quad a = {lo, ll_pair(tag, hi), hi >> 16, tag << 16};
    __builtin_amdgcn_raw_buffer_store_b128(a, B.r, (int)off, 0, kLLAgent);
}

// its value; the tag bits that differ come back in the top half of `wrong`
__device__ __forceinline__ double ll_load1(const LLBuf &B, unsigned off, unsigned tag, unsigned &wrong)
{
    const ll_quad a = __builtin_amdgcn_raw_buffer_load_b128(B.r, (int)off, 0, kLLPoll);
    const unsigned T = tag << 16;
    wrong = (a.y ^ T) | (a.w ^ T);
    return __longlong_as_double((long long)(((ll_word)ll_pair(a.z, a.y) << 32) | a.x));
}

__device__ __forceinline__ bool ll_try1(const LLBuf &B, unsigned off, unsigned tag, double &v)
{
    unsigned wrong;
    v = ll_load1(B, off, tag, wrong);
    return (wrong >> 16) == 0;
}

// One launch's bookkeeping, shared by the kernels' waits.
struct PersistArgs {
    int *status;      // 0, or the number of the first launch that gave up (device memory)
    int *host;        // the same in pinned host memory, written only: the host's to read (or null)
    int launch;       // this launch's number (>= 1)
    unsigned limit;   // polls before a wait gives up
};

__device__ __forceinline__ bool persist_given_up(const PersistArgs &P)
{
    return __hip_atomic_load(P.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// Every lane of the wavefront calls this; attempt() of a lane is true once it
// has its message, each lane polling until then.  False: the wait gave up (the
// same answer in every lane).
template <typename F>
__device__ __forceinline__ bool ll_wait(bool need, const PersistArgs &P, F attempt)
{
    bool ok = !need;
    for (unsigned n = 0;; ++n) {
        if (!ok) ok = attempt();
        if (__all(ok)) return true;
        __builtin_amdgcn_s_sleep(1);
        if ((n & 63u) == 63u && persist_given_up(P)) return false;
        if (n >= P.limit) {
            __hip_atomic_store(P.status, P.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (P.host) __hip_atomic_store(P.host, P.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return false;
        }
    }
}

// Host side.  Resident workgroups of a kernel per CU (0 on error).
int persist_blocks_per_cu(const void *kernel, int threads);
int persist_cus(int device);
unsigned persist_spin_limit();

// Whether a resident form is tried.  Beside much other work on the device a
// launch that gave up will be followed by others, and each costs a wait to its
// bound (about 2 ms); after four in a row the ordinary launches serve the next
// 256 calls (8 us of waiting a call at worst), then the form is tried again.
struct GiveUps {
    int launches = 0, total = 0, inRow = 0, rest = 0;
    bool tries()  // once a call
    {
        if (rest == 0) return true;
        --rest;
        return false;
    }
    void finished() { inRow = 0; }
    void gaveUp()
    {
        ++total;
        if (++inRow >= 4) rest = 256;
    }
};

// Steps of one launch at most: the launches between two settlings stay
// countable, and 3 x steps in an int.
constexpr int kPersistMaxSteps = 1 << 16;

// Launches of resident time steps that are not yet known to have finished, and
// the messages they exchange.  A launch that gave up left its input as it was
// and made the later ones return at once: settle() waits for them and lists the
// runs to do over by ordinary launches.
// The tags of stages count on over the launches.  That a word holds the wanted
// tag or an older one of the last two is true only while every launch writes all
// its messages; after one that gave up, words of any earlier stage are left, and
// 16 bits of tag come round again after 65 536 stages (kPersistMaxSteps steps
// are a multiple of it).  So settle() clears the messages then and the tags
// begin again.
struct ResidentRuns {
    struct Run {
        int launch, first, steps;  // first: steps of the call before this run
        double t0;
        double *in;  // the state the run began with
    };
    // The status word twice: workgroups read it in device memory (in host memory
    // that cost 0.1 us a workgroup), the host in its own (a copy of it took 20 us
    // of each wait for the model).
    int *status = nullptr, *hostStatus = nullptr;
    ll_quad *messages = nullptr;
    size_t messageBytes = 0;
    unsigned tag = 0;              // of the last stage launched; the cleared messages' is 0
    GiveUps ups;
    bool off = false;              // the model does not fit, or there was no memory for its buffers
    std::vector<Run> pending;
    PersistArgs args() const { return {status, hostStatus, ups.launches + 1, persist_spin_limit()}; }
    // call it as soon as the launch is queued: its messages will have been written
    void launched(int first, int steps, double t0, double *in)
    {
        tag += 3u * (unsigned)steps;
        pending.push_back({++ups.launches, first, steps, t0, in});
    }
    int clear(hipStream_t s);      // messages and status, with no launch in flight
    hipError_t alloc_host();
    void free_host();
    int settle(hipStream_t s, std::vector<Run> &again);
};

// Admission of one launch of `blocks` workgroups, `perCu` of which fit a CU.
// The gate keeps the process's resident launches from taking each other's CUs:
// a launch that might not become resident beside the ones in flight on other
// streams is ordered after them.  Construct, check rc, launch, call launched().
class PersistGate {
public:
    PersistGate(int device, hipStream_t stream, int blocks, int perCu);
    int rc;
    int launched();

private:
    std::lock_guard<std::mutex> lock_;
    int device_;
    hipStream_t stream_;
    double demand_, share_;
};

}  // namespace self
