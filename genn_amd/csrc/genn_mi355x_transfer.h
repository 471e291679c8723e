// Part of libgenn_mi355x.so: included by genn_mi355x.hip only (one translation unit).
//
// Copies between host arrays and device arrays in the order of a runner's steps.
//
// What a copy costs here is waiting, not bytes.  hipMemcpy runs on the null stream: behind a kernel on another (blocking)
// stream it takes 41 us for 4 bytes (two queues made to wait for each other), a copy command on the idle stream of its own and a wait
// for it 23 us, and what this file does 9 us (16 behind a step that takes 15 by itself): a copy kernel on the runner's stream that moves the bytes to or from
// pinned host memory and then stores a number the host spins on.
//
// Host arrays that are copied again and again (state, recordings, spike times) are pinned and copied in one
// launch at the rate of PCIe (16 MB: 304 us to the host, 310 from it).  Pinned memory is kept for the next model when a model gives it
// back: touching it for the first time costs 0.4 ms per MiB.  Other host memory goes through a small ring of pinned chunks
// on its way from the device — while the device moves one chunk, the host copies the one before it: 13 MB in 0.5 ms, by
// hipMemcpy 0.8 ms — and by the runtime's own copy on its way there (it reads pageable memory in place: 13 MB in 0.4 ms).
// Where no pinned memory is to be had (GENNMI_PINNED_COPIES=0 asks for none), all of it goes by the runtime's copies.
#ifndef GENN_MI355X_TRANSFER_H
#define GENN_MI355X_TRANSFER_H

namespace
{
constexpr size_t TRANSFER_CHUNK = size_t(1) << 20;      // 18 us of PCIe time: long against a launch, short against a megabyte-sized array
constexpr uint32_t TRANSFER_SLOTS = 4;
constexpr uint32_t TRANSFER_BLOCKS = 32;                // (16 MB from the device with 16 / 32 / 64 / 128 work-groups: 303 / 301 / 302 / 302 us, to it 301 / 311 / 304 / 311)
constexpr size_t PUSH_RING_BYTES = size_t(128) << 10;   // pageable memory up to this size is pushed through the ring (128 KB: 13 us; the runtime takes 20 from there up to 192, 35 for 64)

// Stores that go through to memory.  Nothing then has to be written back before the host (or a kernel on another stream) may look:
// waiting for the stores is enough, where a fence of the whole system in every wavefront made 1 MiB cost 25 us instead of 20.
__device__ __forceinline__ void storeThrough(u32x4 *p, const u32x4 &v) { asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" :: "v"(p), "v"(v) : "memory"); }
template<typename T> __device__ __forceinline__ void storeThrough(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }

// The end of a kernel whose results the host spins for: the work-group that leaves last stores `seq` to the (host) flag.
__device__ __forceinline__ void signalWhenLast(uint32_t *counter, uint32_t *flag, uint32_t seq)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // this thread's stores (storeThrough) have arrived ...
    __syncthreads();                                    // ... and so have the work-group's
    if(threadIdx.x == 0) {
        if(gridDim.x == 1 || atomicAdd(counter, 1u) == gridDim.x - 1) {
            storeThrough(counter, 0u);                  // (for the counter's next user)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            storeThrough(flag, seq);
        }
    }
}

// dst and src have the same offset within 16 bytes
__global__ __launch_bounds__(BLOCK)
void transferKernel(uint8_t *dst, const uint8_t *src, uint32_t bytes, uint32_t *counter, uint32_t *flag, uint32_t seq)
{
    const uint32_t head = min(bytes, (16u - (uint32_t)(reinterpret_cast<uintptr_t>(src) & 15u)) & 15u);
    const uint32_t quads = (bytes - head) / 16;
    const u32x4 *from = reinterpret_cast<const u32x4*>(src + head);
    u32x4 *to = reinterpret_cast<u32x4*>(dst + head);
    const uint32_t thread = blockIdx.x * BLOCK + threadIdx.x, threads = gridDim.x * BLOCK;
    for(uint32_t k = thread; k < quads; k += 4 * threads) {
        u32x4 v[4];
        #pragma unroll
        for(uint32_t u = 0; u < 4; u++) { v[u] = from[min(k + u * threads, quads - 1)]; }
        #pragma unroll
        for(uint32_t u = 0; u < 4; u++) { if(k + u * threads < quads) { storeThrough(to + k + u * threads, v[u]); } }
    }
    if(thread < head) { storeThrough(dst + thread, src[thread]); }
    const uint32_t done = head + 16 * quads;
    if(thread < bytes - done) { storeThrough(dst + done + thread, src[done + thread]); }
    signalWhenLast(counter, flag, seq);
}

// One step's spike queue of every batch: the counts, then `capacity` words per batch that receive as many ids as fit
__global__ __launch_bounds__(BLOCK)
void pullSpikesKernel(const uint32_t *spkCnt, const uint32_t *spk, uint32_t numNeurons, uint32_t slots, uint32_t slot, uint32_t batch, uint32_t capacity,
                      uint32_t *out, uint32_t *counter, uint32_t *flag, uint32_t seq)
{
    for(uint32_t b = blockIdx.x; b < batch; b += gridDim.x) {
        const size_t queue = (size_t)b * slots + slot;
        const uint32_t *ids = spk + queue * numNeurons;
        const uint32_t first = ids[min(threadIdx.x, numNeurons - 1)];      // (asked for with the count: the queue holds numNeurons entries)
        const uint32_t count = min(spkCnt[queue], numNeurons), fit = min(count, capacity);
        uint32_t *to = out + batch + (size_t)b * capacity;
        if(threadIdx.x == 0) { storeThrough(out + b, count); }
        if(threadIdx.x < fit) { storeThrough(to + threadIdx.x, first); }
        for(uint32_t k = threadIdx.x + BLOCK; k < fit; k += BLOCK) { storeThrough(to + k, ids[k]); }
    }
    signalWhenLast(counter, flag, seq);
}

// Elements ahead of the first that lies on 16 bytes in both arrays (all of them: there is none)
__host__ __device__ __forceinline__ size_t copyHead(const float *dst, const float *src, size_t n)
{
    const uintptr_t to = reinterpret_cast<uintptr_t>(dst), from = reinterpret_cast<uintptr_t>(src);
    if(((to ^ from) & 15) || (to & 3)) { return n; }
    return std::min<size_t>(n, ((16 - (to & 15)) & 15) / 4);
}

__global__ __launch_bounds__(BLOCK)
void copySignalKernel(float *dst, const float *src, size_t n, uint32_t *counter, uint32_t *flag, uint32_t seq)
{
    const size_t threads = (size_t)gridDim.x * BLOCK, thread = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    // `count` elements, four of them under way a thread
    auto copy = [&](auto *to, const auto *from, size_t count) {
        for(size_t k = thread; k < count; k += 4 * threads) {
            std::remove_const_t<std::remove_reference_t<decltype(*from)>> v[4];
            #pragma unroll
            for(uint32_t u = 0; u < 4; u++) { v[u] = from[min(k + u * threads, count - 1)]; }
            #pragma unroll
            for(uint32_t u = 0; u < 4; u++) { if(k + u * threads < count) { storeThrough(to + k + u * threads, v[u]); } }
        }
    };
    // quads from the first 16-byte boundary on, where both sides have theirs at the same element
    const size_t head = copyHead(dst, src, n), quads = (n - head) / 4, done = head + 4 * quads;
    copy(reinterpret_cast<u32x4*>(dst + head), reinterpret_cast<const u32x4*>(src + head), quads);
    copy(dst, src, head);
    copy(dst + done, src + done, n - done);
    signalWhenLast(counter, flag, seq);
}

__global__ void signalKernel(uint32_t *flag, uint32_t seq) { storeThrough(flag, seq); }

// How long the host spins for a flag before it blocks instead: a blocking wait wakes up some tens of microseconds after the
// work has ended (GENNMI_POLL_US; 0: block at once)
long pollMicroseconds()
{
    static const long us = [] { const char *e = getenv("GENNMI_POLL_US"); return e ? atol(e) : 2000l; }();
    return us;
}

// Waits until `flag` holds `seq`, which a kernel queued on `stream` stores.  Whatever keeps it from coming (an error of the
// device among them) ends the wait through the blocking call.
int waitForFlag(const uint32_t *flag, uint32_t seq, hipStream_t stream)
{
    const auto begin = std::chrono::steady_clock::now();
    for(uint32_t n = 1; ; n++) {
        if(__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) { return GENNMI_OK; }
        __builtin_ia32_pause();
        if((n & 63u) == 0 && std::chrono::steady_clock::now() - begin > std::chrono::microseconds(pollMicroseconds())) { break; }
    }
    HIP_TRY(hipStreamSynchronize(stream));
    if(__atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq) { HIP_TRY(hipDeviceSynchronize()); }     // (a slot's last user may have been another stream)
    if(__atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq) { return fail(GENNMI_EHIP, "a stream drained without the work that was queued on it"); }
    return GENNMI_OK;
}

// ---- pinned host memory, kept for reuse.  At most PINNED_KEPT bytes lie idle, each block six times as long as idle device memory
// does (genn_mi355x_idle.h): a byte of it takes a thousand times as long to make.  Given back after ten seconds as well, loads
// that far apart took 0.25 ms longer (2.0 against 1.75 of a small network).  What exceeds PINNED_KEPT is given back to the system at
// once, and everything idle is when an allocation fails.
constexpr size_t PINNED_KEPT = size_t(256) << 20, PINNED_UNIT = 4096;
constexpr double PINNED_TIMES = 6.0;
struct PinnedIdle { uintptr_t address; IdleTime until; };
std::mutex g_pinnedMutex;
std::map<uintptr_t, size_t> g_pinned;                   // every block in use or idle: address, bytes
std::multimap<size_t, PinnedIdle> g_pinnedIdle;         // the idle ones by size
size_t g_pinnedIdleBytes = 0;

// (mutex held) gives the idle blocks that are due at `now` back to the system; when the next one is
hipError_t releaseIdlePinned(IdleTime now = IdleTime::max(), IdleTime *next = nullptr)
{
    hipError_t e = hipSuccess;
    for(auto b = g_pinnedIdle.begin(); b != g_pinnedIdle.end(); ) {
        if(b->second.until > now) {
            if(next) { *next = std::min(*next, b->second.until); }
            ++b;
            continue;
        }
        const hipError_t f = hipHostFree(reinterpret_cast<void*>(b->second.address));
        if(f != hipSuccess) { e = f; }
        g_pinned.erase(b->second.address);
        g_pinnedIdleBytes -= b->first;
        b = g_pinnedIdle.erase(b);
    }
    return e;
}

IdleTime pinnedReleaseOld()
{
    std::lock_guard<std::mutex> lock(g_pinnedMutex);
    IdleTime next = IdleTime::max();
    if(releaseIdlePinned(IdleClock::now(), &next) != hipSuccess) { (void)hipGetLastError(); }
    return next;
}

int pinnedMalloc(void **ptr, size_t bytes)
{
    bytes = std::max(PINNED_UNIT, (bytes + PINNED_UNIT - 1) / PINNED_UNIT * PINNED_UNIT);
    std::lock_guard<std::mutex> lock(g_pinnedMutex);
    const auto idle = g_pinnedIdle.lower_bound(bytes);
    if(idle != g_pinnedIdle.end() && idle->first <= bytes + bytes / 4) {
        *ptr = reinterpret_cast<void*>(idle->second.address);
        g_pinnedIdleBytes -= idle->first;
        g_pinnedIdle.erase(idle);
        return GENNMI_OK;
    }
    hipError_t e = hipHostMalloc(ptr, bytes, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable);
    if(e != hipSuccess && !g_pinnedIdle.empty()) {
        (void)hipGetLastError();
        HIP_TRY(releaseIdlePinned());
        e = hipHostMalloc(ptr, bytes, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable);
    }
    if(e != hipSuccess) { (void)hipGetLastError(); }        // (reported here, and not by the next launch of a caller that does without)
    HIP_TRY(e);
    g_pinned[reinterpret_cast<uintptr_t>(*ptr)] = bytes;
    return GENNMI_OK;
}

// false: not a block of this kind
bool pinnedFree(void *ptr, hipError_t *error)
{
    *error = hipSuccess;
    std::lock_guard<std::mutex> lock(g_pinnedMutex);
    const auto block = g_pinned.find(reinterpret_cast<uintptr_t>(ptr));
    if(block == g_pinned.end()) { return false; }
    const IdleTime until = idleUntil(PINNED_TIMES);
    if(g_pinnedIdleBytes + block->second > PINNED_KEPT || until <= IdleClock::now()) {
        g_pinned.erase(block);
        *error = hipHostFree(ptr);
        return true;
    }
    g_pinnedIdle.emplace(block->second, PinnedIdle{block->first, until});
    g_pinnedIdleBytes += block->second;
    releaseIdleAt(until);
    return true;
}

bool isPinned(const void *ptr, size_t bytes)
{
    const uintptr_t a = reinterpret_cast<uintptr_t>(ptr);
    std::lock_guard<std::mutex> lock(g_pinnedMutex);
    auto block = g_pinned.upper_bound(a);
    if(block == g_pinned.begin()) { return false; }
    --block;
    return a + bytes <= block->first + block->second;
}

// A ring of pinned chunks.  Rings are lent to one transfer at a time; a slot is used again when the number its last user
// was given has arrived in its flag.
struct TransferRing
{
    int device = 0;
    uint8_t *chunks = nullptr;          // [TRANSFER_SLOTS][TRANSFER_CHUNK + 16] pinned
    uint32_t *flags = nullptr;          // [TRANSFER_SLOTS][16] pinned, a cache line each
    uint32_t *counters = nullptr;       // [TRANSFER_SLOTS] device memory
    uint32_t seq[TRANSFER_SLOTS] = {};
    uint32_t next = 0;
    uint8_t *chunk(uint32_t slot) const { return chunks + (size_t)slot * (TRANSFER_CHUNK + 16); }
    uint32_t *flag(uint32_t slot) const { return flags + slot * 16; }
};

std::mutex g_ringMutex;
std::vector<TransferRing*> g_rings;     // idle ones; as many exist as transfers have run at once

// copies may take pinned memory of their own (looked at where memory is taken: rings and host sides that exist are used on)
bool pinnedCopies()
{
    const char *e = getenv("GENNMI_PINNED_COPIES");
    return !(e && atoi(e) == 0);
}

// *out: null where there is no memory for a ring
int borrowRing(TransferRing **out)
{
    int device = 0;
    *out = nullptr;
    HIP_TRY(hipGetDevice(&device));
    {
        std::lock_guard<std::mutex> lock(g_ringMutex);
        for(size_t k = 0; k < g_rings.size(); k++) {
            if(g_rings[k]->device == device) { *out = g_rings[k]; g_rings.erase(g_rings.begin() + k); return GENNMI_OK; }
        }
    }
    if(!pinnedCopies()) { return GENNMI_OK; }
    TransferRing *ring = new TransferRing;
    ring->device = device;
    const size_t flagBytes = TRANSFER_SLOTS * 16 * sizeof(uint32_t);
    uint8_t *host = nullptr;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&host), flagBytes + TRANSFER_SLOTS * (TRANSFER_CHUNK + 16), hipHostMallocMapped | hipHostMallocCoherent);
    if(e == hipSuccess) {
        ring->flags = reinterpret_cast<uint32_t*>(host);
        ring->chunks = host + flagBytes;
        memset(host, 0, flagBytes);
        e = hipMalloc(&ring->counters, TRANSFER_SLOTS * sizeof(uint32_t));
    }
    if(e == hipSuccess) { e = hipMemset(ring->counters, 0, TRANSFER_SLOTS * sizeof(uint32_t)); }
    if(e == hipSuccess) { e = hipDeviceSynchronize(); }         // (the counters are cleared before a kernel on any stream uses them)
    if(e != hipSuccess) {
        if(ring->counters) { (void)hipFree(ring->counters); }
        if(host) { (void)hipHostFree(host); }
        delete ring;
        (void)hipGetLastError();
        return GENNMI_OK;           // (an error that is not of this memory comes back from the runtime's copy)
    }
    *out = ring;
    return GENNMI_OK;
}

struct RingLease
{
    TransferRing *ring = nullptr;
    void end()
    {
        if(ring) { std::lock_guard<std::mutex> lock(g_ringMutex); g_rings.push_back(ring); ring = nullptr; }
    }
    ~RingLease() { end(); }
};

// the ring's next slot, once the device is done with what it held
int nextSlot(TransferRing *ring, hipStream_t stream, uint32_t *slot)
{
    *slot = ring->next;
    ring->next = (ring->next + 1) % TRANSFER_SLOTS;
    return waitForFlag(ring->flag(*slot), ring->seq[*slot], stream);
}

// Gives the idle rings back, once the device is done with them
int releaseIdleRings()
{
    std::vector<TransferRing*> rings;
    { std::lock_guard<std::mutex> lock(g_ringMutex); rings.swap(g_rings); }
    int rc = GENNMI_OK, device = 0;
    if(!rings.empty()) { HIP_TRY(hipGetDevice(&device)); }
    for(TransferRing *ring : rings) {
        hipError_t e = hipSetDevice(ring->device);
        if(e == hipSuccess) { e = hipDeviceSynchronize(); }
        if(e == hipSuccess) { e = hipFree(ring->counters); }
        if(e == hipSuccess) { e = hipHostFree(ring->flags); }           // (the chunks lie behind the flags)
        if(e != hipSuccess) { rc = fail(GENNMI_EHIP, std::string("transfer ring: ") + hipGetErrorString(e)); }
        delete ring;
    }
    if(!rings.empty()) { HIP_TRY(hipSetDevice(device)); }
    return rc;
}

struct TransferPart { uint8_t *host; uint8_t *dev; size_t bytes; };

// Splits arrays into chunks: calls chunk(host address, device address, bytes) for each, in order
template<typename F>
int forEachChunk(const TransferPart *parts, uint32_t count, F &&chunk)
{
    for(uint32_t p = 0; p < count; p++) {
        // (pinned memory needs no chunks of the ring, and is the kernel's own source or destination where 16-byte accesses fit both sides)
        const bool direct = ((reinterpret_cast<uintptr_t>(parts[p].host) ^ reinterpret_cast<uintptr_t>(parts[p].dev)) & 15) == 0
                            && isPinned(parts[p].host, parts[p].bytes);
        const size_t most = direct ? size_t(1) << 30 : TRANSFER_CHUNK;
        for(size_t at = 0; at < parts[p].bytes; at += most) {
            const int rc = chunk(parts[p].host + at, parts[p].dev + at, (uint32_t)std::min(most, parts[p].bytes - at), direct);
            if(rc) { return rc; }
        }
    }
    return GENNMI_OK;
}

int launchTransfer(TransferRing *ring, uint32_t slot, uint8_t *dst, const uint8_t *src, uint32_t bytes, hipStream_t stream)
{
    const uint32_t blocks = std::min<uint32_t>(TRANSFER_BLOCKS, std::max<uint32_t>(1, bytes / (16 * BLOCK)));
    transferKernel<<<dim3(blocks), dim3(BLOCK), 0, stream>>>(dst, src, bytes, ring->counters + slot, ring->flag(slot), ring->seq[slot] + 1);
    HIP_TRY(hipGetLastError());
    ring->seq[slot]++;
    return GENNMI_OK;
}

// Device arrays to host arrays, behind everything queued on `stream`; returns when the host arrays hold them
int pullParts(const TransferPart *parts, uint32_t count, hipStream_t stream)
{
    RingLease lease;
    { const int rc = borrowRing(&lease.ring); if(rc) { return rc; } }
    TransferRing *ring = lease.ring;
    if(!ring) {
        for(uint32_t p = 0; p < count; p++) {
            if(parts[p].bytes) { HIP_TRY(hipMemcpyAsync(parts[p].host, parts[p].dev, parts[p].bytes, hipMemcpyDeviceToHost, stream)); }
        }
        HIP_TRY(hipStreamSynchronize(stream));
        return GENNMI_OK;
    }
    struct Pending { uint8_t *host; const uint8_t *chunk; uint32_t bytes, slot, seq; };
    Pending pending[TRANSFER_SLOTS];
    uint32_t first = 0, waiting = 0;
    auto finishOldest = [&]() -> int {
        const Pending &q = pending[first];
        { const int rc = waitForFlag(ring->flag(q.slot), q.seq, stream); if(rc) { return rc; } }
        if(q.chunk) { memcpy(q.host, q.chunk, q.bytes); }
        first = (first + 1) % TRANSFER_SLOTS; waiting--;
        return GENNMI_OK;
    };
    int rc = forEachChunk(parts, count, [&](uint8_t *host, uint8_t *dev, uint32_t bytes, bool direct) -> int {
        if(waiting == TRANSFER_SLOTS) { const int rc2 = finishOldest(); if(rc2) { return rc2; } }
        uint32_t slot;
        { const int rc2 = nextSlot(ring, stream, &slot); if(rc2) { return rc2; } }
        uint8_t *chunk = ring->chunk(slot) + (reinterpret_cast<uintptr_t>(dev) & 15);
        { const int rc2 = launchTransfer(ring, slot, direct ? host : chunk, dev, bytes, stream); if(rc2) { return rc2; } }
        pending[(first + waiting) % TRANSFER_SLOTS] = {host, direct ? nullptr : chunk, bytes, slot, ring->seq[slot]};
        waiting++;
        return GENNMI_OK;
    });
    while(rc == GENNMI_OK && waiting) { rc = finishOldest(); }
    return rc;
}

// Host arrays to device arrays, behind everything queued on `stream`.  The host arrays may be changed as soon as this
// returns; `wait`: so may the device arrays be read, from any stream.
int pushArray(const TransferPart &part, hipStream_t stream, bool wait)
{
    if(part.bytes == 0) { return GENNMI_OK; }
    RingLease lease;
    if(part.bytes <= (wait ? PUSH_RING_BYTES : 2 * TRANSFER_CHUNK) || isPinned(part.host, part.bytes)) { const int rc = borrowRing(&lease.ring); if(rc) { return rc; } }
    TransferRing *ring = lease.ring;
    if(!ring) {
        HIP_TRY(hipMemcpyAsync(part.dev, part.host, part.bytes, hipMemcpyHostToDevice, stream));
        HIP_TRY(hipStreamSynchronize(stream));
        return GENNMI_OK;
    }
    uint32_t last = 0;
    const int rc = forEachChunk(&part, 1, [&](uint8_t *host, uint8_t *dev, uint32_t bytes, bool direct) -> int {
        uint32_t slot;
        { const int rc2 = nextSlot(ring, stream, &slot); if(rc2) { return rc2; } }
        uint8_t *chunk = ring->chunk(slot) + (reinterpret_cast<uintptr_t>(dev) & 15);
        if(!direct) { memcpy(chunk, host, bytes); }
        last = slot;
        wait = wait || direct;
        return launchTransfer(ring, slot, dev, direct ? host : chunk, bytes, stream);
    });
    if(rc || !wait) { return rc; }
    return waitForFlag(ring->flag(last), ring->seq[last], stream);
}

int copyOnDevice(float *dst, const float *src, size_t count, hipStream_t stream)
{
    RingLease lease;
    { const int rc = borrowRing(&lease.ring); if(rc) { return rc; } }
    if(!lease.ring) {
        HIP_TRY(hipMemcpyAsync(dst, src, count * sizeof(float), hipMemcpyDeviceToDevice, stream));
        HIP_TRY(hipStreamSynchronize(stream));
        return GENNMI_OK;
    }
    uint32_t slot;
    { const int rc = nextSlot(lease.ring, stream, &slot); if(rc) { return rc; } }
    // Four quads (elements, where there are no quads) a thread, and no more work-groups than keep memory busy: each ends with an addition to one
    // counter, one after the other, 8 ns each.  Up to 64 work-groups a thread has one of them (30,000 floats 16.4 -> 15.6 us a call).  us a copy
    // with 2048 / 1024 / 512 / 256 / 128 at most: 300,000 floats 12.0 / 11.8 / 12.0 / 11.4 / 10.1, 10^6 19.8 / 19.5 / 14.2 / 11.6 / 11.0, 2.1 x 10^6 32.1
    // / 20.4 / 15.0 / 13.0 / 13.4, 8 x 10^6 34.6 / 23.8 / 18.7 / 19.1 / 25.9, 10^8 175 / 150 / 149 / 201 / 354.  us a call without quads with 2048 / 1024
    // / 512 / 256: 10^6 - / 26.8 / 21.8 / 19.5, 2.1 x 10^6 - / 27.9 / 23.0 / 21.8, 8 x 10^6 42.7 / 32.9 / 31.6 / -, 10^8 169 / 160 / 227 / -; with 2048 and
    // one element a thread under way 27.2, 39.6, 44.0 and 180, with 512 48 and 571 for the last two.
    const bool quads = copyHead(dst, src, count) < count;
    const size_t most = (count <= (size_t(1) << 22)) ? 256 : (quads ? 512 : 1024);
    const size_t one = ((quads ? (count + 3) / 4 : count) + BLOCK - 1) / BLOCK;
    const uint32_t blocks = (uint32_t)std::min<size_t>(most, std::max<size_t>(std::min<size_t>(one, 64), (one + 3) / 4));
    copySignalKernel<<<dim3(blocks), dim3(BLOCK), 0, stream>>>(dst, src, count, lease.ring->counters + slot, lease.ring->flag(slot), lease.ring->seq[slot] + 1);
    HIP_TRY(hipGetLastError());
    lease.ring->seq[slot]++;
    return waitForFlag(lease.ring->flag(slot), lease.ring->seq[slot], stream);
}

// The queue a step left: counts[batch], and the first counts[b] entries of ids[batch][numNeurons]
int pullSpikes(const uint32_t *spkCnt, const uint32_t *spk, uint32_t numNeurons, uint32_t slots, uint32_t slot, uint32_t batch, uint32_t *counts, uint32_t *ids,
               hipStream_t stream)
{
    const size_t words = TRANSFER_CHUNK / sizeof(uint32_t);
    if(batch > words) { return fail(GENNMI_EINVAL, "pull_spikes: too many batches"); }
    auto part = [](uint32_t *host, const uint32_t *dev, size_t count)
    {
        return TransferPart{reinterpret_cast<uint8_t*>(host), reinterpret_cast<uint8_t*>(const_cast<uint32_t*>(dev)), count * sizeof(uint32_t)};
    };
    std::vector<TransferPart> rest;         // queues of more spikes than the chunk holds
    RingLease lease;
    { const int rc = borrowRing(&lease.ring); if(rc) { return rc; } }
    TransferRing *ring = lease.ring;
    if(!ring) {
        for(uint32_t b = 0; b < batch; b++) { rest.push_back(part(counts + b, spkCnt + (size_t)b * slots + slot, 1)); }
        { const int rc = pullParts(rest.data(), batch, stream); if(rc) { return rc; } }
        rest.clear();
        for(uint32_t b = 0; b < batch; b++) {
            counts[b] = std::min(counts[b], numNeurons);
            if(counts[b]) { rest.push_back(part(ids + (size_t)b * numNeurons, spk + ((size_t)b * slots + slot) * numNeurons, counts[b])); }
        }
        return pullParts(rest.data(), (uint32_t)rest.size(), stream);
    }
    const uint32_t capacity = (uint32_t)std::min<size_t>(numNeurons, (words - batch) / batch);
    uint32_t s;
    { const int rc = nextSlot(ring, stream, &s); if(rc) { return rc; } }
    uint32_t *out = reinterpret_cast<uint32_t*>(ring->chunk(s));
    pullSpikesKernel<<<dim3(std::min(batch, TRANSFER_BLOCKS)), dim3(BLOCK), 0, stream>>>(spkCnt, spk, numNeurons, slots, slot, batch, capacity, out,
                                                                                       ring->counters + s, ring->flag(s), ring->seq[s] + 1);
    HIP_TRY(hipGetLastError());
    ring->seq[s]++;
    { const int rc = waitForFlag(ring->flag(s), ring->seq[s], stream); if(rc) { return rc; } }
    memcpy(counts, out, batch * sizeof(uint32_t));
    for(uint32_t b = 0; b < batch; b++) {
        const uint32_t fit = std::min(counts[b], capacity);
        memcpy(ids + (size_t)b * numNeurons, out + batch + (size_t)b * capacity, (size_t)fit * sizeof(uint32_t));
        if(counts[b] > fit) { rest.push_back(part(ids + (size_t)b * numNeurons + fit, spk + ((size_t)b * slots + slot) * numNeurons + fit, counts[b] - fit)); }
    }
    lease.end();
    return rest.empty() ? GENNMI_OK : pullParts(rest.data(), (uint32_t)rest.size(), stream);
}
}   // namespace

#endif
