// devmem.hip -- device memory of short-lived vectors and tables.
//
// A solve allocates its vectors and a potential its tables and fields anew on every call;
// hipMalloc and hipFree of a few hundred MB take 0.1 to several ms each, more than the small
// solves' kernels.  Freed blocks are therefore kept for the next allocation of their size, at
// most kKeep bytes per device, the oldest given back first; all are given back when the last
// context of the device is destroyed, and when any allocation here fails.  A block is kept only
// after the device has finished all work (as hipFree does; or its caller has waited for all that
// used it), so its next owner may use it on any stream.  Contexts in several threads share the list under a
// lock, which no one holds while it waits for the device (hipFree waits too).
#include <list>
#include <mutex>
#include <unordered_map>

#include "mdft_internal.h"

namespace {

constexpr size_t kKeep = (size_t)2 << 30;

struct Block {
    void *p;
    size_t bytes;
    int device;
};
// (never destroyed: a context may be destroyed while the program ends)
std::mutex &lock = *new std::mutex;
std::unordered_map<void *, Block> &live = *new std::unordered_map<void *, Block>;  // allocated through dev_malloc
std::list<Block> &idle = *new std::list<Block>;                                    // oldest first
std::unordered_map<int, int> &users = *new std::unordered_map<int, int>;           // contexts per device

// takes idle blocks of a device off the list, oldest first, until at most `keep` bytes of it are idle (lock held)
std::list<Block> taken(int device, size_t keep) {
    size_t n = 0;
    for (const Block &b : idle)
        if (b.device == device) n += b.bytes;
    std::list<Block> out;
    for (auto it = idle.begin(); it != idle.end() && n > keep;) {
        const auto at = it++;
        if (at->device != device) continue;
        n -= at->bytes;
        out.splice(out.end(), idle, at);
    }
    return out;
}
void give_back(const std::list<Block> &blocks) {
    for (const Block &b : blocks) (void)hipFree(b.p);
}

}  // namespace

hipError_t dev_malloc_bytes(void **p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) bytes = 1;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    {
        const std::lock_guard<std::mutex> hold(lock);
        for (auto it = idle.begin(); it != idle.end(); ++it)
            if (it->device == device && it->bytes == bytes) {
                *p = it->p;
                live[it->p] = *it;
                idle.erase(it);
                return hipSuccess;
            }
    }
    e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        std::list<Block> blocks;
        {
            const std::lock_guard<std::mutex> hold(lock);
            blocks = taken(device, 0);
        }
        give_back(blocks);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();  // told by the return value; the next launch's check is not to find it
        *p = nullptr;
        return e;
    }
    const std::lock_guard<std::mutex> hold(lock);
    live[*p] = Block{*p, bytes, device};
    return hipSuccess;
}

hipError_t dev_free(void *p, bool synced) {
    if (!p) return hipSuccess;
    Block b{};
    bool keep = false;
    {
        const std::lock_guard<std::mutex> hold(lock);
        const auto it = live.find(p);
        if (it != live.end()) {  // else not from dev_malloc
            b = it->second;
            live.erase(it);
            keep = b.bytes <= kKeep && users[b.device] > 0;
        }
    }
    int device = 0;
    keep = keep && hipGetDevice(&device) == hipSuccess && device == b.device &&
           (synced || hipDeviceSynchronize() == hipSuccess);
    if (!keep) return hipFree(p);
    std::list<Block> blocks;
    {
        const std::lock_guard<std::mutex> hold(lock);
        if (users[device] > 0) {
            blocks = taken(device, kKeep - b.bytes);
            idle.push_back(b);
        } else {  // the last context has gone meanwhile
            blocks.push_back(b);
        }
    }
    give_back(blocks);
    return hipSuccess;
}

void dev_context(int device, int change) {
    std::list<Block> blocks;
    {
        const std::lock_guard<std::mutex> hold(lock);
        if ((users[device] += change) <= 0) blocks = taken(device, 0);
    }
    give_back(blocks);
}
