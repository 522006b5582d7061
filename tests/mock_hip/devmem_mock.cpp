// HIP's memory calls on a device of a set size without memory behind it, and devmem.hip's functions with C names:
// the kept device blocks are tested on the CPU.  The calls that wait for the device (hipFree,
// hipDeviceSynchronize) return when the gate is open.
#include <chrono>
#include <condition_variable>
#include <map>
#include <mutex>

#include "mdft_internal.h"

namespace {
std::mutex mu;
std::condition_variable cv;
std::map<void *, size_t> held;
size_t used = 0, room = 0;
uintptr_t next_at = 4096;
int device = 0, waiting = 0;
bool gate = true;
hipError_t last = hipSuccess;

void wait_device() {
    std::unique_lock<std::mutex> l(mu);
    waiting++;
    cv.notify_all();
    cv.wait_for(l, std::chrono::seconds(20), [] { return gate; });
    waiting--;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipDeviceSynchronize() { return wait_device(), hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
    const std::lock_guard<std::mutex> l(mu);
    if (used + n > room) return last = hipErrorOutOfMemory;
    *p = reinterpret_cast<void *>(next_at);
    next_at += (n + 4095) / 4096 * 4096;  // no address is given twice
    held[*p] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    wait_device();
    const std::lock_guard<std::mutex> l(mu);
    if (!held.count(p)) return hipErrorInvalidValue;
    used -= held[p];
    held.erase(p);
    return hipSuccess;
}

void mock_device(int d, size_t bytes) { device = d, room = bytes; }
size_t mock_used() {
    const std::lock_guard<std::mutex> l(mu);
    return used;
}
int mock_holds(void *p) {
    const std::lock_guard<std::mutex> l(mu);
    return (int)held.count(p);
}
void mock_gate(int open) {
    const std::lock_guard<std::mutex> l(mu);
    gate = open != 0;
    cv.notify_all();
}
int mock_await_waiter() {  // 1 once some thread waits for the device
    std::unique_lock<std::mutex> l(mu);
    return cv.wait_for(l, std::chrono::seconds(20), [] { return waiting > 0; }) ? 1 : 0;
}

int t_malloc(void **p, size_t n) { return dev_malloc_bytes(p, n); }
int t_free(void *p, int synced) { return dev_free(p, synced != 0); }
void t_context(int d, int change) { dev_context(d, change); }
}
