// ppmg_readback.hip -- a few device words to the host in the middle of a call.
//
// Every binning ends with the host reading its status words (particles
// outside, overflows, samples), since the launches that follow depend on them.
// A device-to-host copy into pageable memory and a stream synchronisation left
// the device idle for about 55 us (from the end of the key pass to the next
// launch's start, 32^3 cells); a one-workgroup kernel that writes the words and a
// ticket into pinned host memory, on which the host spins, for about 20.  The slots of pinned memory come from one block per process (256
// slots of 1 KiB), one per plan while it lives; a plan that finds none copies.
#include <atomic>
#include <mutex>

#include "ppmg_internal.h"

namespace ppmg {
namespace {

constexpr int SLOT_WORDS = 256;   // the last one is the ticket
constexpr int SLOTS = 256;

std::mutex g_mu;
uint32_t* g_block = nullptr;
bool g_failed = false;
uint64_t g_used[SLOTS / 64] = {};

__global__ void __launch_bounds__(SLOT_WORDS) k_publish(const int* __restrict__ src, int n, uint32_t* dst,
                                                        uint32_t ticket) {
    const int t = threadIdx.x;
    if (t < n) __hip_atomic_store(&dst[t], (uint32_t)src[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (t == 0) __hip_atomic_store(&dst[SLOT_WORDS - 1], ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

uint32_t* host_slot_acquire() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_block) {
        void* p = nullptr;
        if (g_failed || hipHostMalloc(&p, sizeof(uint32_t) * SLOT_WORDS * SLOTS,
                                      hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            g_failed = true;
            return nullptr;
        }
        g_block = static_cast<uint32_t*>(p);
    }
    for (int i = 0; i < SLOTS; ++i)
        if (!((g_used[i / 64] >> (i % 64)) & 1)) {
            g_used[i / 64] |= (uint64_t)1 << (i % 64);
            uint32_t* s = g_block + i * SLOT_WORDS;
            s[SLOT_WORDS - 1] = 0;
            return s;
        }
    return nullptr;
}

void host_slot_release(uint32_t* slot) {
    if (!slot) return;
    std::lock_guard<std::mutex> lk(g_mu);
    const int i = (int)((slot - g_block) / SLOT_WORDS);
    g_used[i / 64] &= ~((uint64_t)1 << (i % 64));
}

// n words at src, as the stream's work before this call leaves them.
int read_back(ppmg_plan* plan, const int* src, int n, int* out, hipStream_t s) {
    if (!plan->host_tried && !arena_bound()) {
        plan->host_tried = true;
        plan->host = host_slot_acquire();
        void* d = nullptr;
        if (plan->host && hipHostGetDevicePointer(&d, plan->host, 0) != hipSuccess) {
            (void)hipGetLastError();
            host_slot_release(plan->host);
            plan->host = nullptr;
        }
        plan->host_dev = static_cast<uint32_t*>(d);
    }
    if (!plan->host || n >= SLOT_WORDS) {
        PPMG_HIP(hipMemcpyAsync(out, src, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost, s));
        PPMG_HIP(hipStreamSynchronize(s));
        return 0;
    }
    if (++plan->ticket == 0) plan->ticket = 1;
    const uint32_t t = plan->ticket;
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(SLOT_WORDS), 0, s, src, n, plan->host_dev, t);
    PPMG_HIP(hipGetLastError());
    auto arrived = [&]() { return __atomic_load_n(&plan->host[SLOT_WORDS - 1], __ATOMIC_ACQUIRE) == t; };
    for (;;) {
        bool got = false;
        for (int i = 0; i < 4096 && !(got = arrived()); ++i) __builtin_ia32_pause();
        if (got) break;
        // now and then ask the stream, so that a failed one ends the wait
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) continue;
        if (e == hipSuccess && arrived()) break;
        PPMG_HIP(hipStreamSynchronize(s));
        if (arrived()) break;
        set_error(PPMG_ERROR_FATAL, PPMG_ERR_DEVICE, "status words did not reach the host");
        return PPMG_ERROR_FATAL;
    }
    for (int i = 0; i < n; ++i) out[i] = (int)plan->host[i];
    return 0;
}

}  // namespace ppmg
