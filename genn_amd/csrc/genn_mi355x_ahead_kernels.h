// Many timesteps of a feed-forward layer per launch (included by genn_mi355x.hip after the synapse and neuron kernels).
//
// A spike source array's spikes depend on nothing but its spike times, and a layer fed by one source alone depends on nothing but
// those spikes: no step of such a network has to wait for the one before it anywhere else than inside a neuron.  The
// reference launches updatePresynapticKernel and updateNeuronsKernel for every step all the same (presynapticUpdateStrategySIMT.cc:
// 57-389, 750-934; backendSIMT.cc:405-662), and so do the step kernels here: each step then pays its launches, the ordered
// spike queue's look-back and a trip of the layer's state through memory.  Here run() takes up to 128 steps at once:
//   1. aheadSourceKernel: a lane walks one source neuron's spikes of all these steps.  Its input to the layer is one 32-bit word per
//      32 steps (bit j: the layer receives a spike from it in step j).
//   2. the layer's input of 32 steps is a matrix product whose left operand is those bits: rows are timesteps, the inner
//      dimension the source neurons (DENSE) or an output pixel's taps (Conv2D), columns the target neurons.
//   3. the neurons: a lane takes one neuron through the steps with its state in registers.
//   4. aheadQueueKernel: the spike queues as the last step leaves them, in ascending neuron index.
// What the next step, of whichever plan, finds is what step-by-step execution leaves: state, queues, recording rows, next spike times.
//
// run() with its launches, copies and waits, one by one -> at once: DENSE 8192 -> 8192 at 5 % activity, 100 steps: 1107 -> 178 us;
// Conv2D 64x64x16 -> 64x64x32 3x3, batch 16, 2.5 %, 50 steps: 2125 -> 795 us, of which 500 move 26 MB between host and device.
#pragma once
#include "genn_mi355x_ahead_layout.h"

namespace
{
constexpr uint32_t AHEAD_MAX_STEPS = 128;                       // steps per pass over the source
constexpr uint32_t AHEAD_DENSE_THREADS = 512, AHEAD_DENSE_WAVES = AHEAD_DENSE_THREADS / WAVE, AHEAD_TILE_COPIES = 4;

struct AheadArgs
{
    unsigned long long timestep, epoch;     // of the first step
    uint32_t steps, batch;
    uint32_t recordingRows;                 // rows of the recording buffers (1: every step writes row 0)
    float dt;
};
struct AheadConv
{
    int32_t kh, kw, ih, iw, ic, oh, ow, oc, PH, PW;
    uint32_t rowsPerBlock, rowPitch, listDepth;         // see AheadConvLayout
    uint32_t isConv;
};

__device__ __forceinline__ size_t aheadRecordingRow(const AheadArgs &A, uint32_t step) { return (size_t)((A.timestep + step) % A.recordingRows); }

// time of a step as the step-by-step path computes it, (float)timestep * dt (a conversion from 64 bits is a dozen instructions; one
// from 32 rounds to the same number, and whether 32 are enough is the same for all steps of a launch)
__device__ __forceinline__ float aheadTime(const AheadArgs &A, uint32_t step)
{
    const bool narrow = ((A.timestep + AHEAD_MAX_STEPS) >> 32) == 0;
    return (narrow ? (float)((uint32_t)A.timestep + step) : (float)(A.timestep + step)) * A.dt;
}

// ---- 1. the source.  Bound by a lane's chain from spike to spike (8192 neurons are 128 wavefronts, each on a SIMD of its own), so that holds few trips
// to memory and few instructions: spike times are asked for SOURCE_AHEAD at a time, while those before are worked off, and a spike's step
// is its time over dt, set right by comparing with the times of the steps around it.  us with a load and a binary search a spike -> now: 100
// steps of 8192 neurons at 5 % 18.8 -> 12.3, 50 steps of 16 x 65,536 at 2.5 % 31.5 -> 20.1 (eight times at once: 13.0 and 20.1).
constexpr uint32_t SOURCE_AHEAD = 4;
__global__ __launch_bounds__(BLOCK)
void aheadSourceKernel(const NeuronGroupDev * __restrict__ source, AheadArgs A, AheadConv C, uint32_t numTrg, uint32_t *words,
                       unsigned long long *eventCounter)
{
    const gennmi_neuron_update_group_t &g = source->g;
    const uint32_t n = g.numNeurons, batch = blockIdx.y, i = blockIdx.x * BLOCK + threadIdx.x, lane = threadIdx.x & (WAVE - 1);
    const size_t bi = (size_t)batch * n + i;
    const uint32_t bitmapWords = (n + 31) / 32;
    uint32_t *recordSpk = g.recordSpk;
    unsigned long long emitted[2] = {0, 0};        // bit k: a spike in the update of step k
    uint32_t queued = 0;                            // ... and in the update before the first
    if(i < n) {
        queued = (asGlobal(source->spikeBitmap)[(A.epoch & 1) * source->bitmapStride + (size_t)batch * bitmapWords + (i >> 5)] >> (i & 31)) & 1u;
        uint32_t start = asGlobal(g.startSpike)[bi];
        const uint32_t end = asGlobal(g.endSpike)[bi], startBefore = start;
        float next = asGlobal(source->nextSpikeTime)[bi];
        GLOBAL_AS const float *times = asGlobal(g.spikeTimes);
        // the times behind the `from`-th of all spikes (nothing is read beyond the neuron's own)
        auto load = [&](uint32_t from, float x[SOURCE_AHEAD]) {
            #pragma unroll
            for(uint32_t u = 0; u < SOURCE_AHEAD; u++) {
                x[u] = INFINITY;
                if(from < end && end - from > u + 1) { x[u] = times[from + u + 1]; }
            }
        };
        float now[SOURCE_AHEAD], later[SOURCE_AHEAD];
        load(start, now);
        const float firstTime = aheadTime(A, 0), lastTime = aheadTime(A, A.steps - 1), perStep = 1.0f / A.dt;
        uint32_t from = 0;
        bool more = true;
        while(more) {
            load(start + SOURCE_AHEAD, later);
            #pragma unroll
            for(uint32_t u = 0; u < SOURCE_AHEAD; u++) {
                // (a NaN is never reached)
                more = more && from < A.steps && lastTime >= next;
                if(more) {
                    // the first step from `from` on whose time has reached the next spike (steps' times ascend)
                    uint32_t step = max(from, (uint32_t)fminf(fmaxf(ceilf((next - firstTime) * perStep), 0.0f), (float)(A.steps - 1)));
                    while(step > from && aheadTime(A, step - 1) >= next) { step--; }
                    while(aheadTime(A, step) < next) { step++; }
                    if(step < 64) { emitted[0] |= 1ull << step; } else { emitted[1] |= 1ull << (step - 64); }
                    start++;
                    // (a start that has passed its end goes on reading, as step by step)
                    next = (start > end) ? times[start] : now[u];
                    from = step + 1;
                }
            }
            #pragma unroll
            for(uint32_t u = 0; u < SOURCE_AHEAD; u++) { now[u] = later[u]; }
        }
        if(start != startBefore) { g.startSpike[bi] = start; source->nextSpikeTime[bi] = next; }
    }
    // the layer's input in step j is what was emitted in the update of step j - 1
    uint32_t received = 0, carry = queued;
    size_t recordingRow = aheadRecordingRow(A, 0);
    #pragma unroll
    for(uint32_t sb = 0; sb < AHEAD_MAX_STEPS / AHEAD_WORD; sb++) {
        if(sb * AHEAD_WORD < A.steps) {
            const uint32_t e = (uint32_t)(emitted[sb / 2] >> (32 * (sb & 1)));
            const uint32_t valid = min(A.steps - sb * AHEAD_WORD, AHEAD_WORD);
            const uint32_t in = ((e << 1) | carry) & (valid == 32 ? 0xFFFFFFFFu : (1u << valid) - 1u);
            carry = e >> 31;
            received += __popc(in);
            if(i < n) { words[((size_t)sb * A.batch + batch) * n + i] = in; }
            // recording rows and the last update's spikes: the wavefront's votes
            if(recordSpk || (sb + 1) * AHEAD_WORD >= A.steps) {
                for(uint32_t j = recordSpk ? 0 : valid - 1; j < valid; j++) {
                    const uint32_t step = sb * AHEAD_WORD + j;
                    const bool last = (step + 1 == A.steps);
                    const unsigned long long ballot = __ballot((e >> j) & 1u);
                    if((lane & 31) == 0 && i < n) {
                        const uint32_t bits = (uint32_t)(ballot >> (lane & 32));
                        if(recordSpk) { recordSpk[(recordingRow * A.batch + batch) * bitmapWords + (i >> 5)] = bits; }
                        // (behind this wavefront's read of the same words; nobody else reads or writes them)
                        if(last) { source->spikeBitmap[((A.epoch + A.steps) & 1) * source->bitmapStride + (size_t)batch * bitmapWords + (i >> 5)] = bits; }
                    }
                    recordingRow = (recordingRow + 1 == A.recordingRows) ? 0 : recordingRow + 1;
                }
            }
        }
    }
    // synaptic events: a dense row has one synapse per target, a pixel of a convolution as many taps as stay inside the output
    unsigned long long events = 0;
    if(received) {
        if(C.isConv) {
            const int pixel = (int)(i / (uint32_t)C.ic), row = pixel / C.iw, col = pixel % C.iw;
            const int firstRow = row - (C.kh - 1 - C.PH), firstCol = col - (C.kw - 1 - C.PW);
            const int rowTaps = min(firstRow + C.kh, C.oh) - max(firstRow, 0), colTaps = min(firstCol + C.kw, C.ow) - max(firstCol, 0);
            events = (unsigned long long)received * (uint32_t)(max(rowTaps, 0) * max(colTaps, 0)) * (uint32_t)C.oc;
        }
        else { events = (unsigned long long)received * numTrg; }
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) { events += __shfl_down(events, off, WAVE); }
    if(lane == 0 && events) { addEvents(eventCounter, events); }
}

// DENSE: the product of 32 steps' bits and 32 columns of weights for 16 sources: v_mfma_f32_32x32x16_bf16 three times.  A bit is 0 or 1, and an
// fp32 weight is exactly the sum of three bfloat16 numbers of 8 significant bits each, so every product is exact, as it is with the fp32
// instruction (v_mfma_f32_32x32x2_f32), which takes eight times 64 clocks for what these three do in 32 each; sums are fp32 either way
// and are rounded less often.  That split needs the lowest of the three to be a normal number and the weight to be finite: weights that are
// not (infinities, NaN, below 2^-90) are multiplied as 0 and added afterwards to the steps that have their spike.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bool aheadOrdinary(float w)
{
    const uint32_t bits = __float_as_uint(w);
    return ((bits & 0x7F800000u) - (37u << 23)) < ((255u - 37u) << 23) || (bits << 1) == 0u;
}
// smallest of eight weights' patterns without sign, moved so that infinities and NaN (from 0), 0 (2^24) and whatever is below 2^-90 lie under
// AHEAD_ORDINARY and all else above: one comparison tells that every one of them can be split as it is
constexpr uint32_t AHEAD_ORDINARY = 38u << 24;
__device__ __forceinline__ uint32_t aheadLeast(const float w[8])
{
    uint32_t q[8];
    #pragma unroll
    for(int k = 0; k < 8; k++) { q[k] = (__float_as_uint(w[k]) << 1) + (1u << 24); }
    return min(min(min(min(q[0], q[1]), q[2]), min(min(q[3], q[4]), q[5])), min(q[6], q[7]));
}
// top 16 bits of two words, packed; what the top 16 bits leave of a float (exact)
__device__ __forceinline__ uint32_t aheadTop(float lower, float upper) { return __builtin_amdgcn_perm(__float_as_uint(upper), __float_as_uint(lower), 0x07060302u); }
__device__ __forceinline__ float aheadRest(float w) { return w - __uint_as_float(__float_as_uint(w) & 0xFFFF0000u); }
// a lane's operand of 8 sources: bit `row` (0..15) of each half of four words as bfloat16 0 or 1
__device__ __forceinline__ bf16x8 aheadBits(u32x4 words, uint32_t row)
{
    u32x4 operand;
    #pragma unroll
    for(int k = 0; k < 4; k++) { operand[k] = ((words[k] >> row) & 0x00010001u) * 0x3F80u; }
    return __builtin_bit_cast(bf16x8, operand);
}
__device__ __forceinline__ f32x16 aheadProduct(bf16x8 bits, bf16x8 weights, f32x16 sum) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bits, weights, sum, 0, 0, 0); }
__device__ __forceinline__ float aheadBit(uint32_t word, uint32_t row) { return (float)((word >> row) & 1u); }
__device__ __forceinline__ bool aheadFinite(float w) { return (__float_as_uint(w) & 0x7F800000u) != 0x7F800000u; }
// the accumulator's element v of a lane in the given half is timestep ...
__device__ __forceinline__ uint32_t aheadRow(uint32_t v, uint32_t half) { return 8 * (v / 4) + 4 * half + (v % 4); }

// ---- 2a. DENSE.  A work-group owns 32 target neurons (columns), up to MT words of (32 steps, batch) as rows and a slice of the
// source; its wavefronts deal the slice's chunks of 64 source neurons among themselves and add their tiles up in LDS in a fixed order.
// Source neurons that are silent in all of the group's steps are dropped first (a ballot packs the others), so what is
// read and multiplied follows the activity: at 5 % and 128 steps all rows remain, at 0.1 % one in eight.  Bound by reading the weights:
// 8192 x 8192 for 100 steps takes 55 us, 4.9 TB/s.  That needs loads under way all the time (75 us where a group's were asked for behind the
// group before it and every chunk began with a trip for its words and one for its first weights) and fewer instructions than the loads leave
// room for: 32-bit offsets of rows in the list instead of 64-bit products, one comparison for eight weights that can be split.  128
// registers: four wavefronts a SIMD.  (152 us with v_mfma_f32_32x32x2_f32, bound by the matrix rate.)  Error of outPost after
// 100 steps against 64 bits, one by one -> here (2-norm, relative): 8192 sources 2.0e-7 -> 1.4e-7, 300 sources 1.6e-7 -> 0.8e-7, weights of
// one sign 1.4e-7 -> 0.7e-7.
template<int MT>
__global__ __launch_bounds__(AHEAD_DENSE_THREADS, 4)
void aheadDenseKernel(const uint32_t * __restrict__ words, uint32_t mTiles, uint32_t mGroups, const float * __restrict__ weights, uint32_t numSrc, uint32_t numTrg,
                      uint32_t sourcesPerSlice, float * __restrict__ partial)
{
    constexpr uint32_t LIST_WORDS = WAVE * (MT + 1), TILE = MT * 32 * 32;
    static_assert(AHEAD_DENSE_WAVES * 2 * LIST_WORDS <= AHEAD_TILE_COPIES * TILE, "lists and tiles share LDS");
    __shared__ __align__(16) uint32_t lds[AHEAD_TILE_COPIES * TILE];
    const uint32_t lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), half = lane >> 5, col = lane & 31;
    const uint32_t mGroup = blockIdx.y % mGroups, slice = blockIdx.y / mGroups;
    const uint32_t firstTile = mGroup * MT;
    const uint32_t column = blockIdx.x * 32 + col, columnByte = min(column, numTrg - 1) * 4, rowBytes = numTrg * 4;
    const uint32_t sliceBegin = slice * sourcesPerSlice, sliceEnd = min(numSrc, sliceBegin + sourcesPerSlice), sliceFirst = sliceBegin + wave * WAVE;
    GLOBAL_AS const uint32_t *in = asGlobal(words);
    // two lists of [64] source neurons, as byte offsets of their rows behind the chunk's first (below 2^32: a layer's input of 32 steps fits
    // AHEAD_MAX_SPACE, and a row is a 32nd of that), then per tile [64] lower and [64] upper halves of their words, 16 bits each
    uint32_t *lists = lds + wave * 2 * LIST_WORDS;
    f32x16 acc[MT];
    #pragma unroll
    for(int q = 0; q < MT; q++) { acc[q] = f32x16{}; }
    auto fetch = [&](uint32_t base, uint32_t mine[MT]) {
        const uint32_t readable = min(base + lane, numSrc - 1);
        #pragma unroll
        for(int q = 0; q < MT; q++) { mine[q] = in[(size_t)min(firstTile + q, mTiles - 1) * numSrc + readable]; }
    };
    // the active ones of 64 source neurons, packed and filled up to a multiple of 16 with entries without spikes; returns how many
    auto pack = [&](uint32_t base, uint32_t mine[MT], uint32_t *list) -> uint32_t {
        uint16_t *halves = reinterpret_cast<uint16_t*>(list + WAVE);
        const uint32_t inside = (base + lane < sliceEnd) ? 0xFFFFFFFFu : 0u;
        uint32_t any = 0;
        #pragma unroll
        for(int q = 0; q < MT; q++) {
            mine[q] &= (firstTile + q < mTiles) ? inside : 0u;
            any |= mine[q];
        }
        const unsigned long long active = __ballot(any != 0);
        const uint32_t count = __popcll(active), filled = (count + 15) / 16 * 16;
        // (a silent one, any of them, fills: it has no bits)
        const uint32_t at = any ? __popcll(active & ((1ull << lane) - 1ull)) : count + __popcll(~active & ((1ull << lane) - 1ull));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");      // (16-bit stores, 128-bit loads: the compiler must not move either across)
        if(at < filled) {
            list[at] = min(lane, sliceEnd - 1 - base) * rowBytes;
            #pragma unroll
            for(int q = 0; q < MT; q++) {
                halves[(2 * q) * WAVE + at] = (uint16_t)mine[q];
                halves[(2 * q + 1) * WAVE + at] = (uint16_t)(mine[q] >> 16);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        return filled;
    };
    auto rowsOf = [&](uint32_t base) { return asGlobal(reinterpret_cast<const char*>(weights + (size_t)base * numTrg)); };
    // Groups of 16 packed sources, a chunk's and then the next one's: a group's weights are asked for before the group ahead of it is worked off, a
    // chunk's words before the chunk ahead of it.  (A chunk's list is made when the last group of the one before is still being read: two lists.)
    uint32_t base = sliceFirst, groups = 0, group = 0, other = 0, mine[MT];
    uint32_t *list = lists;
    GLOBAL_AS const char *rows = nullptr;
    bool special = false;
    // moves on to the next group; false: there is none, and the list's first one stands in for it
    auto advance = [&]() -> bool {
        if(++group < groups) { return true; }
        group = 0;
        uint32_t found = 0;
        while(base < sliceEnd && found == 0) {
            found = pack(base, mine, lists + other) / 16;
            base += AHEAD_DENSE_THREADS;
            fetch(base, mine);
        }
        if(found == 0) { return false; }
        groups = found;
        rows = rowsOf(base - AHEAD_DENSE_THREADS);
        list = lists + other;
        other = LIST_WORDS - other;
        return true;
    };
    auto load = [&](float x[8]) {
        const u32x4 *sources = reinterpret_cast<const u32x4*>(list) + 4 * group + 2 * half;
        const u32x4 first = sources[0], second = sources[1];
        #pragma unroll
        for(int k = 0; k < 4; k++) {
            x[k] = *reinterpret_cast<GLOBAL_AS const float*>(rows + (first[k] + columnByte));
            x[4 + k] = *reinterpret_cast<GLOBAL_AS const float*>(rows + (second[k] + columnByte));
        }
    };
    // works the group off whose weights are in b, those of the next one on their way into `following`; false: it was the last
    auto work = [&](float b[8], float following[8]) -> bool {
        // a lane's rows are the steps of its column number: the lower or the upper halves
        const u32x4 *bits = reinterpret_cast<const u32x4*>(list + WAVE + (col >> 4) * (WAVE / 2)) + half + 2 * group;
        const bool more = advance();
        load(following);            // (not behind a branch: b is then waited for while these are under way)
        if(__ballot(aheadLeast(b) < AHEAD_ORDINARY)) {
            #pragma unroll
            for(int k = 0; k < 8; k++) {
                const bool ordinary = aheadOrdinary(b[k]);
                special = special || !ordinary;
                b[k] = ordinary ? b[k] : 0.0f;
            }
        }
        u32x4 top, middle, low;
        #pragma unroll
        for(int k = 0; k < 4; k++) {
            const float r0 = aheadRest(b[2 * k]), r1 = aheadRest(b[2 * k + 1]);
            top[k] = aheadTop(b[2 * k], b[2 * k + 1]);
            middle[k] = aheadTop(r0, r1);
            low[k] = aheadTop(aheadRest(r0), aheadRest(r1));
        }
        bf16x8 a[MT];
        #pragma unroll
        for(int q = 0; q < MT; q++) { a[q] = aheadBits(bits[q * (WAVE / 4)], col & 15); }
        #pragma unroll
        for(int q = 0; q < MT; q++) { acc[q] = aheadProduct(a[q], __builtin_bit_cast(bf16x8, low), acc[q]); }
        #pragma unroll
        for(int q = 0; q < MT; q++) { acc[q] = aheadProduct(a[q], __builtin_bit_cast(bf16x8, middle), acc[q]); }
        #pragma unroll
        for(int q = 0; q < MT; q++) { acc[q] = aheadProduct(a[q], __builtin_bit_cast(bf16x8, top), acc[q]); }
        return more;
    };
    fetch(base, mine);
    if(advance()) {
        float even[8], odd[8];
        load(even);
        while(work(even, odd) && work(odd, even)) {}
    }
    if(__ballot(special)) {
        for(base = sliceFirst; base < sliceEnd; base += AHEAD_DENSE_THREADS) {
            fetch(base, mine);
            const uint32_t count = pack(base, mine, lists);
            const uint16_t *halves = reinterpret_cast<const uint16_t*>(lists + WAVE);
            for(uint32_t k = 0; k < count; k++) {
                const float x = *reinterpret_cast<GLOBAL_AS const float*>(rowsOf(base) + (lists[k] + columnByte));
                if(aheadOrdinary(x)) { continue; }
                #pragma unroll
                for(int q = 0; q < MT; q++) {
                    const uint32_t word = halves[(2 * q) * WAVE + k] | ((uint32_t)halves[(2 * q + 1) * WAVE + k] << 16);
                    #pragma unroll
                    for(uint32_t v = 0; v < 16; v++) { acc[q][v] += ((word >> aheadRow(v, half)) & 1u) ? x : 0.0f; }
                }
            }
        }
    }
    // ---- the wavefronts' tiles: four copies in LDS, two rounds, then the sum of the copies
    float *tiles = reinterpret_cast<float*>(lds);
    float *copy = tiles + (wave % AHEAD_TILE_COPIES) * TILE;
    #pragma unroll
    for(uint32_t round = 0; round < AHEAD_DENSE_WAVES / AHEAD_TILE_COPIES; round++) {
        __syncthreads();
        if(wave / AHEAD_TILE_COPIES == round) {
            #pragma unroll
            for(int q = 0; q < MT; q++) {
                #pragma unroll
                for(uint32_t v = 0; v < 16; v++) {
                    float *e = &copy[(q * 32 + aheadRow(v, half)) * 32 + col];
                    *e = round ? *e + acc[q][v] : acc[q][v];
                }
            }
        }
    }
    __syncthreads();
    for(uint32_t e = threadIdx.x; e < TILE; e += AHEAD_DENSE_THREADS) {
        const uint32_t tile = firstTile + e / 1024, row = (e / 32) % 32, j = blockIdx.x * 32 + e % 32;
        if(tile < mTiles && j < numTrg) {
            partial[(((size_t)slice * mTiles + tile) * 32 + row) * numTrg + j] = (tiles[e] + tiles[TILE + e]) + (tiles[2 * TILE + e] + tiles[3 * TILE + e]);
        }
    }
}

// What a target neuron needs of its group, and one of its steps: postsynaptic model on outPost plus the step's input, current
// source, neuron model (operations and order of neuronBulkBody).  Neuron and postsynaptic model are known when the kernel is compiled:
// the steps are unrolled, and a branch on either would be taken in each of them.
template<uint32_t MODEL, uint32_t PSM, bool SELECT = false>
struct AheadNeuron
{
    PlainNeuron constants;
    float psmInit, psmDecay, inject, dt;
    __device__ __forceinline__ explicit AheadNeuron(const gennmi_neuron_update_group_t &g, float timestep)
        : constants(plainNeuronOf(g)), psmInit(g.psm[0].init), psmDecay(g.psm[0].expDecay), inject(g.numCS ? g.cs[0].amp : 0.0f), dt(timestep)
    {
        constants.model = MODEL;
    }
    __device__ __forceinline__ bool step(float input, float &linSyn, float &v0, float &v1) const
    {
        float Isyn = 0;
        linSyn += input;
        if(PSM == GENNMI_PSM_EXPCURR) {
            Isyn += psmInit * linSyn;
            linSyn *= psmDecay;
        }
        else {
            Isyn += linSyn;
            linSyn = 0.0f;
        }
        Isyn += inject;         // (a sum that starts at +0 is never -0: adding +0 where there is no source changes nothing)
        return SELECT ? selected(Isyn, v0, v1) : plainNeuronStep(constants, Isyn, dt, v0, v1);
    }
    // plainNeuronStep with a LIF neuron's two paths both computed: what does not depend on V is then off the chain from step to step
    __device__ __forceinline__ bool selected(float Isyn, float &v0, float &v1) const
    {
        if(MODEL != GENNMI_NEURON_LIF) { return plainNeuronStep(constants, Isyn, dt, v0, v1); }
        const float alpha = ((Isyn + constants.p[0]) * constants.p[1]) + constants.p[2];
        const bool free = (v1 <= 0.0f);
        float moved = alpha - (constants.p[3] * (alpha - v0)), waited = v1 - dt;
        asm volatile("" : "+v"(moved), "+v"(waited));       // (the compiler would make a branch around them again)
        v0 = free ? moved : v0;
        v1 = free ? v1 : waited;
        const bool spiked = (v1 <= 0.0f && v0 >= constants.p[4]);
        v0 = spiked ? constants.p[5] : v0;
        v1 = spiked ? constants.p[6] : v1;
        return spiked;
    }
};

// ---- 3a. the neurons behind a DENSE projection: one lane each, 16 steps' inputs asked for while the 16 before are worked off (a
// population of 8192 is 128 wavefronts: the chain of steps bounds it, so work-groups are single wavefronts, spread over the chip).
// The 16 steps are straight code (both paths of a LIF neuron computed, votes kept in a register, stored once a group): 100 steps of 8192
// neurons 21.4 us with a branch for the refractory neurons, the last step and the recorder in every step, 16.4 without.  The compiler had put the
// branch back and waited for a group's inputs as soon as it had asked for them, to add up the slices: with both paths kept apart from that, and one
// or two slices added up when they are used (SLICES), 16.6 -> 13.2 us.
template<uint32_t MODEL, uint32_t PSM, uint32_t SLICES>
__global__ __launch_bounds__(WAVE)
void aheadNeuronKernel(const NeuronGroupDev * __restrict__ target, AheadArgs A, const float * __restrict__ partial, uint32_t slices, uint32_t mTiles, uint32_t *lastBits)
{
    const gennmi_neuron_update_group_t &g = target->g;
    const uint32_t n = g.numNeurons, batch = blockIdx.y, lane = threadIdx.x, i = blockIdx.x * WAVE + lane;
    const uint32_t bitmapWords = (n + 31) / 32;
    AheadNeuron<MODEL, PSM, true> neuron(g, A.dt);
    asm volatile("" : "+v"(neuron.constants.p[5]), "+v"(neuron.constants.p[6]));       // (selected between in every step: from scalar registers that is a copy first)
    const size_t bi = (size_t)batch * n + min(i, n - 1);
    uint32_t *recordSpk = g.recordSpk;
    constexpr uint32_t GROUP = 16;
    GLOBAL_AS float *var0 = asGlobal(g.var0), *var1 = asGlobal(g.var1), *outPost = asGlobal(g.psm[0].outPost);
    float v0 = var0[bi], v1 = var1[bi], lin = outPost[bi];
    GLOBAL_AS const float *input = asGlobal(partial) + min(i, n - 1);
    // a group's inputs, on their way where the source is cut into one or two slices (added up when they are used), or already added up
    struct Inputs { float x[GROUP], y[SLICES == 2 ? GROUP : 1]; };
    auto load = [&](uint32_t first, Inputs &to) {
        const size_t row = ((size_t)(first / 32) * A.batch + batch) * 32 + first % 32, slice = (size_t)mTiles * 32;
        if(SLICES != 0) {
            #pragma unroll
            for(uint32_t u = 0; u < GROUP; u++) {
                to.x[u] = input[(row + u) * n];
                if(SLICES == 2) { to.y[u] = input[(row + slice + u) * n]; }
            }
            return;
        }
        #pragma unroll
        for(uint32_t u = 0; u < GROUP; u++) { to.x[u] = 0.0f; }
        #pragma unroll 2
        for(uint32_t k = 0; k < slices; k++) {
            #pragma unroll
            for(uint32_t u = 0; u < GROUP; u++) { to.x[u] += input[(k * slice + row + u) * n]; }
        }
    };
    auto inputOf = [&](const Inputs &from, uint32_t u) {
        const float x = (SLICES == 0) ? from.x[u] : 0.0f + from.x[u];
        return (SLICES == 2) ? x + from.y[u] : x;
    };
    // A step's votes go to two lanes of `votes`, and a group's steps leave with one store: lane u (16 + u) has the lower (upper) word of step u.
    const unsigned long long present = __builtin_amdgcn_ballot_w64(i < n);
    const uint32_t voteStep = lane & 15, voteWord = (blockIdx.x * WAVE >> 5) + ((lane >> 4) & 1);
    const bool voteLane = lane < 32 && voteWord < bitmapWords;
    // (`all`: 1, and the steps of the group are one straight piece of code; 0: some of them are beyond the last)
    auto group = [&](uint32_t first, const Inputs &now, auto all) {
        uint32_t votes = 0;
        #pragma unroll
        for(uint32_t u = 0; u < GROUP; u++) {
            if(all.value || first + u < A.steps) {
                const unsigned long long ballot = __builtin_amdgcn_ballot_w64(neuron.step(inputOf(now, u), lin, v0, v1)) & present;
                votes = (voteStep == u) ? ((lane & 16) ? (uint32_t)(ballot >> 32) : (uint32_t)ballot) : votes;
            }
        }
        const uint32_t step = first + voteStep;
        if(voteLane && step < A.steps) {
            // (of the steps of this launch that share a recording row only the last writes it)
            if(recordSpk && A.steps - step <= A.recordingRows) { recordSpk[(aheadRecordingRow(A, step) * A.batch + batch) * bitmapWords + voteWord] = votes; }
            if(step + 1 == A.steps) { lastBits[(size_t)batch * bitmapWords + voteWord] = votes; }
        }
    };
    // (two groups' inputs that change places, not values)
    auto work = [&](uint32_t first, const Inputs &now, Inputs &next) -> bool {
        if(first + GROUP < A.steps) { load(first + GROUP, next); }
        if(first + GROUP <= A.steps) { group(first, now, std::integral_constant<uint32_t, 1>()); }
        else { group(first, now, std::integral_constant<uint32_t, 0>()); }
        return first + GROUP < A.steps;
    };
    Inputs even, odd;
    load(0, even);
    for(uint32_t first = 0; work(first, even, odd) && work(first + GROUP, odd, even); first += 2 * GROUP) {}
    if(i < n) { var0[bi] = v0; var1[bi] = v1; outPost[bi] = lin; }
}

// 32 x 32 bits per half-wave, transposed by exchanging ever smaller blocks across the diagonal.  A lane's neighbours are reached without LDS, and a block is
// moved by a rotation and put in place by a bit select: 17 instructions.
struct Transpose32
{
    uint32_t keep[5], turn[5];
    __device__ __forceinline__ explicit Transpose32(uint32_t lane)
    {
        // (low: the bits b with b & j == 0; a lane with lane & j keeps the others and takes its neighbour's, moved down)
        constexpr uint32_t low[5] = {0x0000FFFFu, 0x00FF00FFu, 0x0F0F0F0Fu, 0x33333333u, 0x55555555u};
        #pragma unroll
        for(uint32_t k = 0; k < 5; k++) {
            const uint32_t j = 16u >> k;
            keep[k] = (lane & j) ? ~low[k] : low[k];
            turn[k] = (lane & j) ? j : 32u - j;
        }
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t x) const
    {
        const auto rows = __builtin_amdgcn_permlane16_swap(x, x, false, false);             // the lower row's and the upper row's, in both
        exchange<0>(x, (keep[0] == 0xFFFF0000u) ? rows[0] : rows[1]);
        exchange<1>(x, dpp<0x128>(x));                                                      // row_ror:8
        exchange<2>(x, dpp<0x1B>(dpp<0x141>(x)));                                           // row_half_mirror, quad_perm:[3,2,1,0]
        exchange<3>(x, dpp<0x4E>(x));                                                       // quad_perm:[2,3,0,1]
        exchange<4>(x, dpp<0xB1>(x));                                                       // quad_perm:[1,0,3,2]
        return x;
    }
private:
    template<int K>
    __device__ __forceinline__ void exchange(uint32_t &x, uint32_t other) const
    {
        const uint32_t turned = __builtin_amdgcn_alignbit(other, other, turn[K]);
        x = (x & keep[K]) | (turned & ~keep[K]);
    }
    template<int CTRL>
    static __device__ __forceinline__ uint32_t dpp(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xF, 0xF, false); }
};

// ---- 2b, 3b. Conv2D and its neurons, up to 32 steps.  A work-group owns some output rows of one batch and 32 output channels: the
// words of the input pixels they reach (zero outside the input) and the kernel wait in LDS.  A wavefront takes two output pixels at a
// time: the rows of its two products are timesteps, the inner dimension the pixel's (tap, channel) inputs that have a spike in any of the
// steps, packed into a list in LDS in their order (45 % of them are silent at 2.5 % activity and 32 steps).  The products stay in registers; one
// swap of half-wavefronts per register pair puts a neuron's 32 inputs into one lane, which takes the neuron through the steps and leaves
// its spikes as one word.
// The products are those of the step kernel, v_mfma_f32_32x32x2_f32 over taps and channels in the same order, which adds one input after
// the other: leaving out inputs whose bits are all 0 changes no bit of a sum, whichever two then share an instruction, so a layer's sums are
// the same bits whether its steps are taken at once or one by one.  (With weights in three bfloat16 parts, as in aheadDenseKernel, one spike in
// 10^6 moves by a step.)
// us for 32 steps of 64x64x16 -> 64x64x32 3x3, batch 16, at 2.5 %: 198 with pairs left out that are silent together and a weight read once for
// four pixels, 183 packed with a branch around each product (the sixteen sums are copied wherever the paths meet), 144 packed and straight.
// Of that the matrix cores are busy 60 and the vector units 64 (counters), the neurons' steps half of these.  run() with all its launches, packed
// against paired, other shapes and rates: 40x37x16 -> 4 5x5 batch 16, 32 steps, 0.5 / 5 / 40 / 100 % 124 / 248 / 385 / 422 against 244 / 398 / 481 / 507; 24x24x16 -> 32
// 5x5, 45 steps 96 / 165 / 270 / 298 against 189 / 283 / 358 / 375; the shape above, 50 steps 179 / 318 / 549 / 746 against 243 / 416 / 586 / 771.
// Where few of a pixel's inputs have a spike in a step (2.5 %: 3.6 of 144), most of a product's rows add nothing, and a sum is made one weight after the
// other instead, in the same order and so with the same bits: the words of 32 inputs, transposed, give each lane one step's, which it lists in LDS, and the
// pixel's lanes add up the weights listed for step after step, four at a time.  A product of two inputs is 64 clocks of the matrix unit whatever they hold;
// a listed weight is two or three vector instructions, so the rule (aheadConvMost) compares 48 clocks an active input with 48 a step, 300 a transposed word and 6 a
// spike, and leaves to the products patches of more spikes a pixel and step than 13/32 of what a list holds (6.5 where it holds 16; one that is full means products
// for its two pixels).  A list holds a quarter of the inputs, 16 at most, and no more than leaves a compute unit its work-groups (aheadConvLayout).
// run() of 50 steps, products only -> now, at 0.5 / 2.5 / 10 / 30 / 75 %: 64x64x16 -> 32 3x3 batch 16 196 / 308 / 440 / 540 / 687 -> 197 / 235 / 440 / 540 / 687; 48x48x3 ->
// 20 5x5 batch 8 90 / 116 / 145 / 164 / 172 -> 89 / 108 / 144 / 164 / 172; 40x37x16 -> 4 5x5 batch 16, 24x24x16 -> 32 5x5 batch 4, 64x64 from one channel, 33x47x2: no change; 64x72x16 -> 32 3x3
// batch 16, at 0.5 / 2.5 / 10 / 30 %, lists of 12: 206 / 329 / 500 / 620 -> 205 / 253 / 498 / 620.
template<uint32_t MODEL, uint32_t PSM>
__global__ __launch_bounds__(BLOCK, 4)
void aheadConvKernel(const NeuronGroupDev * __restrict__ target, AheadArgs A, AheadConv C, uint32_t wordBlock, const uint32_t * __restrict__ words,
                     const float * __restrict__ kernel, uint32_t *spikeWords)
{
    extern __shared__ __align__(16) uint32_t shAhead[];
    const gennmi_neuron_update_group_t &g = target->g;
    const uint32_t n = g.numNeurons, batch = blockIdx.y, oc = (uint32_t)C.oc, ow = (uint32_t)C.ow;
    const uint32_t lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), half = lane >> 5, col = lane & 31;
    const uint32_t y0 = blockIdx.x * C.rowsPerBlock, rows = min(C.rowsPerBlock, (uint32_t)C.oh - y0), pixels = rows * ow;
    const uint32_t o = blockIdx.z * 32 + col;
    const uint32_t steps = min(A.steps - wordBlock * AHEAD_WORD, AHEAD_WORD);
    AheadNeuron<MODEL, PSM> neuron(g, A.dt);
    asm volatile("" : "+v"(neuron.constants.p[5]), "+v"(neuron.constants.p[6]));       // (selected between in every step: from scalar registers that is a copy first)
    const uint32_t rowPitch = C.rowPitch, rowWords = (uint32_t)(C.kw * C.ic), inputs = (uint32_t)C.kh * rowWords;
    const uint32_t depth = C.listDepth, quads = depth / 4, listBytes = aheadConvListBytes(inputs, depth), zeroRow = depth ? 1u : 0u;
    uint8_t *lists = reinterpret_cast<uint8_t*>(shAhead) + wave * listBytes;
    uint2 *list = reinterpret_cast<uint2*>(lists);                                                  // (word, byte of its weights) of a pixel's active inputs
    uint16_t *stepList = reinterpret_cast<uint16_t*>(lists);                                        // [pixel][step][depth] bytes of weights
    float *kern = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(shAhead) + (BLOCK / WAVE) * listBytes);     // [input][32], with lists of steps one more of zeros
    uint16_t *place = reinterpret_cast<uint16_t*>(kern + (inputs + zeroRow) * 32);                        // [input] its word behind the pixel's first
    uint32_t *patch = reinterpret_cast<uint32_t*>(kern + (inputs + zeroRow) * 32) + (inputs + 1) / 2;
    // ---- the patch: row r, word e is word e - PW * ic of input row y0 - PH + r
    GLOBAL_AS const uint32_t *in = asGlobal(words) + ((size_t)wordBlock * A.batch + batch) * ((size_t)C.ih * C.iw * C.ic);
    const int inRowWords = C.iw * C.ic;
    uint32_t active = 0, spiked = 0;
    for(uint32_t r = 0; r < rows + (uint32_t)C.kh - 1; r++) {
        const int y = (int)(y0 + r) - C.PH;
        for(uint32_t e = threadIdx.x; e < rowPitch; e += BLOCK) {
            const int x = (int)e - C.PW * C.ic;
            const uint32_t word = (y >= 0 && y < C.ih && x >= 0 && x < inRowWords) ? in[(size_t)y * inRowWords + x] : 0u;
            patch[r * rowPitch + e] = word;
            active += (word != 0u) ? 1u : 0u;
            spiked += __popc(word);
        }
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) { active += __shfl_down(active, off, WAVE); spiked += __shfl_down(spiked, off, WAVE); }
    __shared__ uint32_t seen[2][BLOCK / WAVE];
    if(lane == 0) { seen[0][wave] = active; seen[1][wave] = spiked; }
    bool nonFinite = false;
    for(uint32_t e = threadIdx.x; e < (inputs + zeroRow) * 32; e += BLOCK) {
        const uint32_t k = e / 32, oo = blockIdx.z * 32 + (e & 31);
        float weight = (oo < oc && k < inputs) ? asGlobal(kernel)[(size_t)k * oc + oo] : 0.0f;
        if(!aheadFinite(weight)) { nonFinite = true; weight = 0.0f; }
        kern[e] = weight;
    }
    for(uint32_t k = threadIdx.x; k < inputs; k += BLOCK) { place[k] = (uint16_t)(k / rowWords * rowPitch + k % rowWords); }
    nonFinite = __syncthreads_or(nonFinite);

    GLOBAL_AS float *var0 = asGlobal(g.var0) + (size_t)batch * n, *var1 = asGlobal(g.var1) + (size_t)batch * n, *outPost = asGlobal(g.psm[0].outPost) + (size_t)batch * n;
    GLOBAL_AS uint32_t *spikes = asGlobal(spikeWords) + (size_t)batch * n;
    const char *weights = reinterpret_cast<const char*>(kern + col);
    const uint2 *entries = list + half;
    // Lists, for each of 32 steps, the inputs that have a spike in it, in their order: lane (half, t) those of the half's pixel in step t.  32 inputs at a
    // time, a lane each, their words transposed.  false: a step has more than `most`.
    active = spiked = 0;
    #pragma unroll
    for(uint32_t w = 0; w < BLOCK / WAVE; w++) { active += seen[0][w]; spiked += seen[1][w]; }
    // (of the patch's words those that are input: a work-group at the edge has no more to add up for most of its pixels than any other)
    const int firstRow = max((int)y0 - C.PH, 0), endRow = min((int)(y0 + rows) + C.kh - 1 - C.PH, C.ih), firstWord = max(C.PW * C.ic, 0), endWord = min(C.PW * C.ic + inRowWords, (int)rowPitch);
    const uint32_t inputWords = (uint32_t)max(endRow - firstRow, 0) * (uint32_t)max(endWord - firstWord, 0);
    const uint32_t most = nonFinite ? 0u : aheadConvMost(depth, inputs, steps, active, spiked, inputWords);
    const Transpose32 transposed(lane);
    auto listSteps = [&](uint32_t pixel, uint32_t &count) -> bool {
        auto word = [&](uint32_t k) -> uint32_t {
            const uint32_t there = patch[pixel + place[min(k, inputs - 1)]];
            return (k < inputs) ? there : 0u;
        };
        uint32_t bits = word(col), following = word(32 + col);
        bits = transposed(bits);
        uint16_t *mine = stepList + lane * depth;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for(uint32_t q = 0; q < quads; q++) { reinterpret_cast<u32x2*>(mine)[q] = u32x2{inputs * 0x800080u, inputs * 0x800080u}; }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for(uint32_t k0 = 0; ; ) {
            if(__ballot(count + __popc(bits) > most)) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                return false;
            }
            while(bits) {
                mine[count++] = (uint16_t)((k0 + __ffs(bits) - 1) * 128);
                bits &= bits - 1;
            }
            k0 += 32;
            if(k0 >= inputs) { break; }
            bits = transposed(following);
            following = word(k0 + 32 + col);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        return true;
    };
    for(uint32_t first = wave * 2; first < pixels; first += (BLOCK / WAVE) * 2) {
        // state of the lane's neuron (pixel first + half, channel o), asked for ahead of the products
        const uint32_t own = first + half;
        const bool valid = (own < pixels && o < oc);
        const size_t at = valid ? ((size_t)y0 * ow + own) * oc + o : 0;
        float v0 = var0[at], v1 = var1[at], lin = outPost[at];
        uint32_t base[2];
        #pragma unroll
        for(int j = 0; j < 2; j++) {
            const uint32_t p = min(first + j, pixels - 1), r = p / ow;
            base[j] = r * rowPitch + (p - r * ow) * (uint32_t)C.ic;
        }
        // (kept a comparison and a branch: computed ahead for all steps, the conditions are 32 masks, spilled)
        uint32_t fired = 0, count = 0;
        auto step = [&](uint32_t t, float input) {
            uint32_t end = steps;
            asm volatile("" : "+s"(end));
            if(t < end) {
                asm volatile("" : "+v"(lin));
                fired |= neuron.step(input, lin, v0, v1) ? 1u << t : 0u;
            }
        };
        if(most != 0 && listSteps(half ? base[1] : base[0], count)) {
            // four of a step's inputs at a time, both halves as many rounds as the one that has more needs
            uint32_t more[AHEAD_CONV_MOST / 4];
            #pragma unroll
            for(uint32_t q = 0; q < AHEAD_CONV_MOST / 4; q++) {
                const unsigned long long ballot = __ballot(count > 4 * q);
                more[q] = (uint32_t)ballot | (uint32_t)(ballot >> 32);
            }
            const u32x2 *mine = reinterpret_cast<const u32x2*>(stepList + half * AHEAD_WORD * depth);
            auto load = [&](u32x2 four, float w[4]) {
                w[0] = *reinterpret_cast<const float*>(weights + (four[0] & 0xFFFFu)); w[1] = *reinterpret_cast<const float*>(weights + (four[0] >> 16));
                w[2] = *reinterpret_cast<const float*>(weights + (four[1] & 0xFFFFu)); w[3] = *reinterpret_cast<const float*>(weights + (four[1] >> 16));
            };
            // (the first four of a group of steps are asked for ahead of the group before; a loop, for the instruction cache's sake)
            constexpr uint32_t GROUP = 4;
            float w[GROUP][4], next[GROUP][4];
            #pragma unroll
            for(uint32_t u = 0; u < GROUP; u++) { load(mine[u * quads], w[u]); }
            #pragma unroll 1
            for(uint32_t t0 = 0; t0 < steps; t0 += GROUP) {
                const uint32_t ahead = min(t0 + GROUP, AHEAD_WORD - GROUP);
                #pragma unroll
                for(uint32_t u = 0; u < GROUP; u++) { load(mine[(ahead + u) * quads], next[u]); }
                __builtin_amdgcn_sched_barrier(0);
                #pragma unroll
                for(uint32_t u = 0; u < GROUP; u++) {
                    const uint32_t t = t0 + u;
                    float input = (((0.0f + w[u][0]) + w[u][1]) + w[u][2]) + w[u][3];
                    #pragma unroll
                    for(uint32_t q = 1; q < AHEAD_CONV_MOST / 4; q++) {
                        if(!((more[q] >> t) & 1u)) { break; }
                        float x[4];
                        load(mine[t * quads + q], x);
                        input = (((input + x[0]) + x[1]) + x[2]) + x[3];
                    }
                    step(t, input);
                }
                #pragma unroll
                for(uint32_t u = 0; u < GROUP; u++) {
                    #pragma unroll
                    for(uint32_t k = 0; k < 4; k++) { w[u][k] = next[u][k]; }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        else {
            f32x16 acc[2];
            #pragma unroll
            for(int j = 0; j < 2; j++) {
                acc[j] = f32x16{};
                // the inputs that have a spike in any of the steps, in their order
                uint32_t count = 0;
                for(uint32_t k0 = 0; k0 < inputs; k0 += WAVE) {
                    const uint32_t k = k0 + lane;
                    const uint32_t behind = place[min(k, inputs - 1)], there = patch[base[j] + behind], word = (k < inputs) ? there : 0u;
                    const unsigned long long active = __ballot(word != 0u);
                    if(word) { list[count + __popcll(active & ((1ull << lane) - 1ull))] = make_uint2(word, k * 128); }
                    count += __popcll(active);
                }
                if(lane == 0) { list[count] = make_uint2(0u, 0u); }         // (fills the last pair)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                // (no branch inside a round: the compiler copies the sixteen sums where paths with and without a product meet)
                uint32_t m = 0;
                for(; m + 8 <= count; m += 8) {
                    uint2 e[4]; float w[4];
                    #pragma unroll
                    for(uint32_t u = 0; u < 4; u++) { e[u] = entries[m + 2 * u]; }
                    #pragma unroll
                    for(uint32_t u = 0; u < 4; u++) { w[u] = *reinterpret_cast<const float*>(weights + e[u].y); }
                    #pragma unroll
                    for(uint32_t u = 0; u < 4; u++) { acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(aheadBit(e[u].x, col), w[u], acc[j], 0, 0, 0); }
                }
                for(; m < count; m += 2) {
                    const uint2 e = entries[m];
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(aheadBit(e.x, col), *reinterpret_cast<const float*>(weights + e.y), acc[j], 0, 0, 0);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
            if(nonFinite) {
                // weights that are not finite, to the steps that have their spike only (see aheadDenseKernel)
                for(uint32_t k = 0; k < inputs; k++) {
                    const float b = (o < oc) ? asGlobal(kernel)[(size_t)k * oc + o] : 0.0f;
                    if(aheadFinite(b)) { continue; }
                    #pragma unroll
                    for(int j = 0; j < 2; j++) {
                        const uint32_t bits = patch[base[j] + place[k]];
                        #pragma unroll
                        for(uint32_t v = 0; v < 16; v++) { acc[j][v] += ((bits >> aheadRow(v, half)) & 1u) ? b : 0.0f; }
                    }
                }
            }
            // lower half: all steps of the first pixel, upper half: of the second
            float x[16], y[16];
            #pragma unroll
            for(int v = 0; v < 16; v++) {
                const auto swapped = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][v]), __float_as_uint(acc[1][v]), false, false);
                x[v] = __uint_as_float(swapped[0]); y[v] = __uint_as_float(swapped[1]);
            }
            #pragma unroll
            for(uint32_t t = 0; t < AHEAD_WORD; t++) { step(t, (t & 4) ? y[4 * (t / 8) + (t & 3)] : x[4 * (t / 8) + (t & 3)]); }
        }
        if(valid) { var0[at] = v0; var1[at] = v1; outPost[at] = lin; spikes[at] = fired; }
    }
}

// (the kernel of the target's neuron model and postsynaptic model)
template<uint32_t SLICES>
auto aheadNeuronInstance(const gennmi_neuron_update_group_t &g)
{
    constexpr uint32_t LIF = GENNMI_NEURON_LIF, IZH = GENNMI_NEURON_IZHIKEVICH, EXP = GENNMI_PSM_EXPCURR, DELTA = GENNMI_PSM_DELTACURR;
    const bool lif = (g.model == LIF), exponential = (g.psm[0].kind == EXP);
    return lif ? (exponential ? aheadNeuronKernel<LIF, EXP, SLICES> : aheadNeuronKernel<LIF, DELTA, SLICES>)
               : (exponential ? aheadNeuronKernel<IZH, EXP, SLICES> : aheadNeuronKernel<IZH, DELTA, SLICES>);
}

// The layer's spikes turned from one word per neuron (32 steps) into one word per step (32 neurons): the recording rows and the bitmap of
// the last step.  A work-group takes 1024 neurons so that a step's words leave as 128 consecutive bytes.
__global__ __launch_bounds__(BLOCK)
void aheadTransposeKernel(const NeuronGroupDev * __restrict__ target, AheadArgs A, uint32_t wordBlock, const uint32_t * __restrict__ spikeWords, uint32_t *lastBits)
{
    __shared__ uint32_t rows[AHEAD_WORD][33];
    const gennmi_neuron_update_group_t &g = target->g;
    const uint32_t n = g.numNeurons, batch = blockIdx.y, lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const uint32_t steps = min(A.steps - wordBlock * AHEAD_WORD, AHEAD_WORD), bitmapWords = (n + 31) / 32;
    uint32_t mine[4];
    #pragma unroll
    for(uint32_t q = 0; q < 4; q++) {
        const uint32_t i = blockIdx.x * 1024 + (wave * 4 + q) * WAVE + lane;
        mine[q] = (i < n) ? asGlobal(spikeWords)[(size_t)batch * n + i] : 0u;
    }
    const Transpose32 transposed(lane);
    #pragma unroll
    for(uint32_t q = 0; q < 4; q++) {
        // (32 ballots and selects instead: 18 us for 2.1 x 10^6 neurons)
        rows[lane & 31][(wave * 4 + q) * 2 + (lane >> 5)] = transposed(mine[q]);
    }
    __syncthreads();
    for(uint32_t e = threadIdx.x; e < AHEAD_WORD * 32; e += BLOCK) {
        const uint32_t t = e / 32, word = blockIdx.x * 32 + e % 32, step = wordBlock * AHEAD_WORD + t;
        if(t >= steps || word >= bitmapWords) { continue; }
        // (of the steps of this launch that share a recording row only the last writes it)
        if(g.recordSpk && steps - t <= A.recordingRows) { g.recordSpk[(aheadRecordingRow(A, step) * A.batch + batch) * bitmapWords + word] = rows[t][e % 32]; }
        if(step + 1 == A.steps) { lastBits[(size_t)batch * bitmapWords + word] = rows[t][e % 32]; }
    }
}

// ---- 4. the queues of both populations from the bitmaps of the last step: a work-group per population and batch, its threads
// own consecutive words, so a scan of their counts is the ascending order
constexpr uint32_t AHEAD_QUEUE_THREADS = 1024;
__global__ __launch_bounds__(AHEAD_QUEUE_THREADS)
void aheadQueueKernel(const NeuronGroupDev * __restrict__ populations, const uint32_t *sourceBits, const uint32_t *targetBits)
{
    __shared__ uint32_t waveTotal[AHEAD_QUEUE_THREADS / WAVE];
    const gennmi_neuron_update_group_t &g = populations[blockIdx.x].g;
    const uint32_t n = g.numNeurons, words = (n + 31) / 32, batch = blockIdx.y, lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    GLOBAL_AS const uint32_t *bits = asGlobal(blockIdx.x ? targetBits : sourceBits) + (size_t)batch * words;
    GLOBAL_AS uint32_t *queue = asGlobal(g.spk) + (size_t)batch * n;
    const uint32_t per = (words + AHEAD_QUEUE_THREADS - 1) / AHEAD_QUEUE_THREADS;
    const uint32_t begin = min(threadIdx.x * per, words), end = min(begin + per, words);
    uint32_t mine = 0;
    for(uint32_t w = begin; w < end; w++) { mine += __popc(bits[w]); }
    uint32_t scan = mine;
    for(int off = 1; off < WAVE; off <<= 1) { const uint32_t up = __shfl_up(scan, off, WAVE); if(lane >= (uint32_t)off) { scan += up; } }
    if(lane == WAVE - 1) { waveTotal[wave] = scan; }
    __syncthreads();
    uint32_t position = scan - mine, total = 0;
    for(uint32_t w = 0; w < AHEAD_QUEUE_THREADS / WAVE; w++) {
        if(w < wave) { position += waveTotal[w]; }
        total += waveTotal[w];
    }
    for(uint32_t w = begin; w < end; w++) {
        uint32_t word = bits[w];
        while(word) {
            const uint32_t bit = __ffs(word) - 1;
            word &= word - 1;
            queue[position++] = w * 32 + bit;
        }
    }
    if(threadIdx.x == 0) { g.spkCnt[batch] = total; }
}
}   // namespace
