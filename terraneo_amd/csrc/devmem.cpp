// Device memory of the library's own objects (operators' matrices, multigrid
// vectors, Krylov workspaces), with a bounded cache of freed blocks.
//
// A program replaces these objects all the time -- new operators and a new
// hierarchy with every viscosity field, a workspace with every solve -- and
// hipMalloc / hipFree of the same sizes cost more than the work: at lateral
// level 6 the set-up after a new viscosity spent 4 to 40 ms of its 22 to 41 ms
// there (mapping, and the driver clearing released memory), a Stokes step at
// level 4 allocates 30 vectors.
//
// Rules:
//  * a freed block may still be read by work in flight on any stream, so a block
//    freed since the device's last synchronisation here is handed out only after
//    a device synchronisation (what hipFree did at every free);
//  * destroying an object, and the end of a solve, wait for the device (dev_wait),
//    also as hipFree did: the caller may free or overwrite its own arrays then;
//  * at most 1/16 of the device's memory is cached, the rest is freed at once;
//  * the cache is emptied when an allocation of the library fails (then retried),
//    when the last live block of the device is freed and on dev_trim, by which the
//    host program gets it back for its own allocator.
// Blocks belong to the device they were allocated on; all calls are serialised
// by one mutex, so any thread may allocate and free.
#include <map>
#include <mutex>
#include <unordered_map>

#include "tn_internal.hpp"

namespace tn {
namespace {

struct DeviceCache {
    std::multimap<size_t, void*> free_blocks;  // by class size
    size_t cached = 0, limit = 0;
    int64_t live = 0;
    bool dirty = false;  // a cached block was freed after the last synchronisation
};
struct Block {
    size_t bytes;
    int device;
};
struct Pool {
    std::mutex mu;
    std::map<int, DeviceCache> dev;
    std::unordered_map<void*, Block> live;
};
// never destroyed: objects may be freed while the process ends
Pool& pool()
{
    static Pool* p = new Pool;
    return *p;
}

// Size classes, so that a slightly different size finds a block: powers of two
// to 1 MiB, eight per octave to 256 MiB, above that multiples of 2 MiB (large
// arrays waste nothing).
size_t class_size(size_t bytes)
{
    constexpr size_t MiB = size_t(1) << 20;
    if (bytes > 256 * MiB) return (bytes + 2 * MiB - 1) / (2 * MiB) * (2 * MiB);
    size_t p = 512;
    while (p < bytes) p <<= 1;
    if (bytes <= MiB) return p;
    const size_t step = p / 16;  // p / 2 < bytes <= p
    return (bytes + step - 1) / step * step;
}

void release(DeviceCache& c)
{
    for (auto& b : c.free_blocks) (void)hipFree(b.second);
    c.free_blocks.clear();
    c.cached = 0;
    c.dirty = false;
}

}  // namespace

void* dev_alloc(size_t bytes)
{
    if (bytes == 0) return nullptr;
    int device = 0;
    TN_HIP(hipGetDevice(&device));
    const size_t size = class_size(bytes);
    Pool& p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    DeviceCache& c = p.dev[device];
    void* ptr = nullptr;
    auto it = c.free_blocks.find(size);
    if (it != c.free_blocks.end()) {
        if (c.dirty) {
            TN_HIP(hipDeviceSynchronize());
            c.dirty = false;
        }
        ptr = it->second;
        c.free_blocks.erase(it);
        c.cached -= size;
    } else {
        hipError_t e = hipMalloc(&ptr, size);
        if (e == hipErrorOutOfMemory && !c.free_blocks.empty()) {
            (void)hipGetLastError();
            release(c);
            e = hipMalloc(&ptr, size);
        }
        TN_HIP(e);
    }
    p.live.emplace(ptr, Block{size, device});
    ++c.live;
    return ptr;
}

void dev_free(void* ptr)
{
    if (!ptr) return;
    Pool& p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    auto it = p.live.find(ptr);
    if (it == p.live.end()) return;
    const Block b = it->second;
    p.live.erase(it);
    DeviceCache& c = p.dev[b.device];
    --c.live;
    if (c.limit == 0) {
        hipDeviceProp_t prop;
        c.limit = hipGetDeviceProperties(&prop, b.device) == hipSuccess ? prop.totalGlobalMem / 16 : 1;
    }
    if (c.cached + b.bytes > c.limit) {
        (void)hipFree(ptr);
    } else {
        c.free_blocks.emplace(b.bytes, ptr);
        c.cached += b.bytes;
        c.dirty = true;
    }
    if (c.live == 0) release(c);
}

void dev_wait()
{
    std::vector<int> held;
    {
        Pool& p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        for (const auto& d : p.dev)
            if (d.second.live > 0) held.push_back(d.first);
    }
    int current = 0;
    if (held.empty() || hipGetDevice(&current) != hipSuccess) return;
    for (int d : held) {
        if (d != current) (void)hipSetDevice(d);
        (void)hipDeviceSynchronize();
        if (d != current) (void)hipSetDevice(current);
    }
}

// Pinned pages: a solve takes one; freed pages are kept (as many as were ever in
// use at once) until dev_trim.
namespace {
struct Pages {
    std::mutex mu;
    std::vector<double*> idle;
};
Pages& pages()
{
    static Pages* p = new Pages;
    return *p;
}
}  // namespace

HostPage::HostPage() : p(nullptr)
{
    {
        std::lock_guard<std::mutex> lk(pages().mu);
        if (!pages().idle.empty()) {
            p = pages().idle.back();
            pages().idle.pop_back();
            return;
        }
    }
    TN_HIP(hipHostMalloc((void**)&p, HOST_PAGE_BYTES, hipHostMallocPortable));
}

HostPage::~HostPage()
{
    std::lock_guard<std::mutex> lk(pages().mu);
    pages().idle.push_back(p);
}

void dev_trim()
{
    {
        Pool& p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        for (auto& d : p.dev) release(d.second);  // (hipFree waits for the block's device)
    }
    std::vector<double*> idle;
    {
        std::lock_guard<std::mutex> lk(pages().mu);
        idle.swap(pages().idle);
    }
    for (double* q : idle) (void)hipHostFree(q);
}

}  // namespace tn
