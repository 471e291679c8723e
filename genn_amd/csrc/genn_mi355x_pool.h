// Part of libgenn_mi355x.so: included by genn_mi355x.hip only (one translation unit).
//
// Device memory that is kept when a model gives it back.  hipMalloc and hipFree of a gigabyte take 0.3 ms each, and once as
// much memory as the card holds has been freed, 20 ms: the driver clears what it hands out again.  A program that builds
// model after model (a parameter scan, a session) paid that for every one of them.  Unloading a model of 10^5 neurons with 10^8 synapses
// and loading the next of the same sizes takes 1.4 ms from kept blocks and 3.7 ms where no kept block fits (GENNMI_POOL_SECONDS=0).
//
// Blocks of POOL_SMALLEST bytes and more are kept, at most a thirty-second of the card's memory in all, and each for ten seconds
// (GENNMI_POOL_SECONDS; 0: none is kept), after which a thread of the library's gives it back, also in a process that does
// nothing any more; an allocation that fails gives all of them back first, and gennmi_release_cached_memory does at any time.
// A kept block is handed out again only after everything that the device had been given when the block was freed has
// finished, on whatever stream and from whatever thread.
#ifndef GENN_MI355X_POOL_H
#define GENN_MI355X_POOL_H

namespace
{
constexpr size_t POOL_SMALLEST = size_t(2) << 20;           // (smaller ones the runtime hands out in less than a microsecond)

struct DevicePool
{
    struct Idle { void *ptr; size_t bytes; int device; bool finished; IdleTime until; };
    struct Used { size_t bytes; int device; };
    std::mutex mutex;
    std::map<void*, Used> used;
    std::vector<Idle> idle;             // in the order they were freed
    size_t idleBytes = 0, limit = 0;

    // (mutex held)
    hipError_t release(size_t k)
    {
        const Idle block = idle[k];
        idleBytes -= block.bytes;
        idle.erase(idle.begin() + k);
        return hipFree(block.ptr);
    }
    hipError_t releaseAll()
    {
        hipError_t e = hipSuccess;
        while(!idle.empty()) { const hipError_t f = release(idle.size() - 1); if(f != hipSuccess) { e = f; } }
        return e;
    }
    hipError_t releaseOld()
    {
        const IdleTime now = IdleClock::now();
        for(size_t k = 0; k < idle.size(); ) {
            if(idleBytes <= limit && idle[k].until > now) { k++; continue; }
            const hipError_t e = release(k);
            if(e != hipSuccess) { return e; }
        }
        return hipSuccess;
    }
};
DevicePool g_pool;

// (called by the library's thread) gives back what has been idle long enough; when to look again
IdleTime poolReleaseOld()
{
    std::lock_guard<std::mutex> lock(g_pool.mutex);
    const IdleTime now = IdleClock::now();
    IdleTime next = IdleTime::max();
    for(size_t k = 0; k < g_pool.idle.size(); ) {
        if(g_pool.idle[k].until > now) { next = std::min(next, g_pool.idle[k++].until); continue; }
        if(hipSetDevice(g_pool.idle[k].device) != hipSuccess) { (void)hipGetLastError(); k++; continue; }
        if(g_pool.release(k) != hipSuccess) { (void)hipGetLastError(); }
    }
    return next;
}

hipError_t poolMalloc(void **ptr, size_t bytes)
{
    if(bytes < POOL_SMALLEST) { return hipMalloc(ptr, bytes); }
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if(e != hipSuccess) { return e; }
    std::lock_guard<std::mutex> lock(g_pool.mutex);
    e = g_pool.releaseOld();
    if(e != hipSuccess) { return e; }
    size_t best = g_pool.idle.size();
    for(size_t k = 0; k < g_pool.idle.size(); k++) {
        const auto &b = g_pool.idle[k];
        if(b.device == device && b.bytes >= bytes && b.bytes <= bytes + bytes / 8 && (best == g_pool.idle.size() || b.bytes < g_pool.idle[best].bytes)) { best = k; }
    }
    if(best != g_pool.idle.size()) {
        if(!g_pool.idle[best].finished) {
            e = hipDeviceSynchronize();         // (as hipFree would have done when the block was given back)
            if(e != hipSuccess) { return e; }
            for(auto &b : g_pool.idle) { b.finished = b.finished || b.device == device; }
        }
        const auto block = g_pool.idle[best];
        g_pool.idleBytes -= block.bytes;
        g_pool.idle.erase(g_pool.idle.begin() + best);
        g_pool.used[block.ptr] = {block.bytes, device};
        *ptr = block.ptr;
        return hipSuccess;
    }
    e = hipMalloc(ptr, bytes);
    if(e != hipSuccess && !g_pool.idle.empty()) {
        (void)hipGetLastError();
        e = g_pool.releaseAll();
        if(e == hipSuccess) { e = hipMalloc(ptr, bytes); }
    }
    if(e == hipSuccess) { g_pool.used[*ptr] = {bytes, device}; }
    return e;
}
template<typename T> hipError_t poolMalloc(T **ptr, size_t bytes) { return poolMalloc(reinterpret_cast<void**>(ptr), bytes); }

hipError_t poolFree(void *ptr)
{
    if(!ptr) { return hipSuccess; }
    {
        std::lock_guard<std::mutex> lock(g_pool.mutex);
        const auto block = g_pool.used.find(ptr);
        if(block != g_pool.used.end()) {
            if(g_pool.limit == 0) {
                size_t freeBytes = 0, total = 0;
                const hipError_t e = hipMemGetInfo(&freeBytes, &total);
                if(e != hipSuccess) { return e; }
                g_pool.limit = total / 32;
            }
            const IdleTime until = idleUntil();
            g_pool.idle.push_back({ptr, block->second.bytes, block->second.device, false, until});
            g_pool.idleBytes += block->second.bytes;
            g_pool.used.erase(block);
            const hipError_t e = g_pool.releaseOld();
            if(!g_pool.idle.empty()) { releaseIdleAt(until); }
            return e;
        }
    }
    return hipFree(ptr);
}

// memory an allocation could get: what the device has left and what is kept here
hipError_t poolFreeBytes(size_t *bytes)
{
    size_t total = 0;
    const hipError_t e = hipMemGetInfo(bytes, &total);
    if(e != hipSuccess) { return e; }
    int device = 0;
    const hipError_t f = hipGetDevice(&device);
    std::lock_guard<std::mutex> lock(g_pool.mutex);
    for(const auto &b : g_pool.idle) { if(b.device == device) { *bytes += b.bytes; } }
    return f;
}
}   // namespace

#endif
