// Part of libgenn_mi355x.so: included by genn_mi355x.hip only (one translation unit).
#ifndef GENN_MI355X_NEURON_KERNELS_H
#define GENN_MI355X_NEURON_KERNELS_H

namespace
{
// State a step leaves behind goes through the L2 to memory at once: what is dirty when a kernel ends is written back then, and the next
// kernel waits for it.  us a step, written back at the end / through: 10^6 Izhikevich neurons 20.8 / 20.1, the microcircuit at 35 % with PoissonExp
// sources, a launch a step, 7.5 / 7.25, 100,000 neurons with plastic synapses 20.4 / 20.0; 300,000 LIF neurons 13.1 / 13.0, no more than two runs differ.
template<typename T>
__device__ __forceinline__ void storeThrough(GLOBAL_AS T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// PoissonExp current source (currentSourceModels.h:100-129): the snippet's loop draws uniforms until their product falls to
// ExpMinusLambda; here the draws of (neuron, step) are the words of counter-based generator calls, so the result does not
// depend on the launch geometry or on which plan steps the network.
__device__ __forceinline__ uint32_t poissonExpCount(const gennmi_cs_t &cs, size_t bi, unsigned long long epoch)
{
    const gennmi_rows::Stream s{(uint32_t)cs.seed, (uint32_t)(cs.seed >> 32), cs.stream};
    float p = 1.0f;
    uint32_t numSpikes = 0;
    for(uint32_t call = 0; ; call++) {
        const gennmi_rows::Words r = gennmi_rows::philox4x32((uint32_t)bi, (uint32_t)epoch, call, s.stream, s.k0, s.k1);
        bool done = false;
        #pragma unroll
        for(int w = 0; w < 4 && !done; w++) {
            numSpikes++;
            p *= gennmi_rows::uniformHalfOpen(r.w[w]);
            done = !(p > cs.expMinusLambda);
        }
        if(done) { break; }
    }
    return numSpikes - 1;
}

// one step of the source whose state the caller holds: returns the injected value, leaves the decayed one in `current`
__device__ __forceinline__ float poissonExpStep(const gennmi_cs_t &cs, float &current, size_t bi, unsigned long long epoch)
{
    const float value = current + cs.init * (float)poissonExpCount(cs, bi, epoch);
    current = value * cs.expDecay;
    return value;
}

__device__ __forceinline__ float poissonExpInject(const gennmi_cs_t &cs, GLOBAL_AS float *current, size_t bi, unsigned long long epoch)
{
    float state = current[bi];
    const float value = poissonExpStep(cs, state, bi, epoch);
    current[bi] = state;
    return value;
}

// ------------------------------------------------------------------------------------------------
// Sum of the counts of the earlier blocks of a population, by all threads of a block with every count asked for at once; all threads get it.
// 0xFFFFFFFF after a bounded wait expired (error flag raised).
// ------------------------------------------------------------------------------------------------
// Populations of more blocks than a wavefront has lanes and of no more than this: one trip after the last count instead of the three of two
// levels (counts of the group, its total out, totals in).  Beyond, a step in which every block has spikes would read more counts than spikes.
// Counts that have not arrived at the first look are asked for again together; eight at once instead of four cost registers (300,000 neurons 6.0 -> 8.5).
// us a step of neurons alone, two levels -> counts asked for again one by one -> together, no spike / one in 20,000 / one in 200 of the neurons: 20,000
// neurons 4.64 -> 4.36 -> 4.34, 4.67 -> 4.42 -> 4.38, 4.89 -> 4.58 -> 4.58; 140,000 4.73 -> 4.80 -> 4.78, 5.03 -> 4.83 -> 4.78, 6.12 -> 5.02 -> 4.99; 300,000
// 5.40 -> 5.70 -> 5.54, 5.67 -> 5.82 -> 5.67, 7.07 -> 6.01 -> 5.84; 520,000 7.25 -> 7.40 -> 7.31, 7.66 -> 7.57 -> 7.46, 10.87 -> 8.23 -> 8.07.
constexpr uint32_t QUEUE_DIRECT_BLOCKS = 2048, COUNTS_AT_ONCE = 4;
__host__ __device__ __forceinline__ bool queueDirect(uint32_t numBlocks) { return numBlocks > WAVE && numBlocks <= QUEUE_DIRECT_BLOCKS; }
__device__ __forceinline__ uint32_t sumOfEarlierBlocks(uint32_t localBlock, const unsigned long long *counts, uint32_t tag, uint32_t *errorFlag)
{
    __shared__ uint32_t shSum[1024 / WAVE];
    const uint32_t lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, threads = blockDim.x;
    uint32_t sum = 0, spins = 0;
    bool ok = true;
    for(uint32_t first = 0; first < localBlock && ok; first += COUNTS_AT_ONCE * threads) {
        unsigned long long word[COUNTS_AT_ONCE];
        uint32_t pending = 0;
        // (a count that is not there to be read: 0 with the step's tag)
        #pragma unroll
        for(uint32_t u = 0; u < COUNTS_AT_ONCE; u++) {
            const uint32_t k = first + u * threads + threadIdx.x;
            word[u] = (unsigned long long)tag << 32;
            if(k < localBlock) { word[u] = __hip_atomic_load(&counts[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
        }
        // (those that had not arrived are asked for again together, not one after the other)
        while(true) {
            pending = 0;
            #pragma unroll
            for(uint32_t u = 0; u < COUNTS_AT_ONCE; u++) { pending |= ((uint32_t)(word[u] >> 32) != tag) ? 1u << u : 0u; }
            if(pending == 0) { break; }
            if(++spins > c_spinLimit) { ok = false; break; }
            __builtin_amdgcn_s_sleep(1);
            #pragma unroll
            for(uint32_t u = 0; u < COUNTS_AT_ONCE; u++) {
                if((pending >> u) & 1u) { word[u] = __hip_atomic_load(&counts[first + u * threads + threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
            }
        }
        #pragma unroll
        for(uint32_t u = 0; u < COUNTS_AT_ONCE; u++) { sum += (uint32_t)word[u]; }
    }
    if(!ok) { raiseErrorFlag(errorFlag); }
    for(int off = WAVE / 2; off > 0; off >>= 1) { sum += __shfl_down(sum, off, WAVE); }
    if(lane == 0) { shSum[wave] = sum; }
    const bool allOk = (__syncthreads_and(ok) != 0);
    sum = 0;
    for(uint32_t w = 0; w < threads / WAVE; w++) { sum += shSum[w]; }
    return allOk ? sum : 0xFFFFFFFFu;
}

// ------------------------------------------------------------------------------------------------
// Offset of a block's entries in its population's queue: the block publishes its count, then (wave 0) sums the counts of
// the earlier blocks of its group of 64 and the published totals of the earlier groups.  Every thread of the block calls
// this between two barriers of its own; returns 0xFFFFFFFF after a bounded wait expired (error flag raised).
// (`published`: the caller has stored the block's count itself, earlier — see publishBlockCount)
__device__ __forceinline__ void publishBlockCount(uint32_t blockCount, uint32_t localBlock, size_t aggBase, unsigned long long *counts, uint32_t tag)
{
    if(threadIdx.x == 0) {
        __hip_atomic_store(&counts[aggBase + localBlock], ((unsigned long long)tag << 32) | blockCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
template<bool DIRECT = true>
__device__ __forceinline__ uint32_t blockQueueOffset(uint32_t blockCount, uint32_t localBlock, uint32_t numBlocks, size_t aggBase,
                                                    unsigned long long *counts, unsigned long long *groupTotals, uint32_t tag,
                                                    uint32_t *shOffset, uint32_t *errorFlag, bool published = false)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t wave = threadIdx.x / WAVE;
    if(threadIdx.x == 0 && !published) {
        __hip_atomic_store(&counts[aggBase + localBlock], ((unsigned long long)tag << 32) | blockCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool last = (localBlock == numBlocks - 1);
    if(DIRECT && queueDirect(numBlocks)) {
        // (a block without spikes that is not the last needs no offset)
        return (blockCount != 0 || last) ? sumOfEarlierBlocks(localBlock, counts + aggBase, tag, errorFlag) : 0u;
    }
    if(wave == 0) {
        const uint32_t group = localBlock / WAVE, inGroup = localBlock % WAVE;
        const size_t groupBase = aggBase + (size_t)group * WAVE;
        bool ok = true;
        auto waitFor = [&](const unsigned long long *p) -> uint32_t {
            uint32_t spins = 0;
            while(true) {
                const unsigned long long a = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if((uint32_t)(a >> 32) == tag) { return (uint32_t)a; }
                if(++spins > c_spinLimit) { ok = false; return 0u; }
                __builtin_amdgcn_s_sleep(1);
            }
        };
        uint32_t intra = (lane < inGroup) ? waitFor(&counts[groupBase + lane]) : 0u;
        for(int off = WAVE / 2; off > 0; off >>= 1) { intra += __shfl_down(intra, off, WAVE); }
        intra = __shfl(intra, 0, WAVE);
        if((inGroup == WAVE - 1 || last) && lane == 0 && ok) {
            __hip_atomic_store(&groupTotals[aggBase + group], ((unsigned long long)tag << 32) | (intra + blockCount), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        uint32_t sum = 0;
        if(blockCount != 0 || last) {
            for(uint32_t base = 0; base < group; base += WAVE) {
                if(base + lane < group) { sum += waitFor(&groupTotals[aggBase + base + lane]); }
            }
            for(int off = WAVE / 2; off > 0; off >>= 1) { sum += __shfl_down(sum, off, WAVE); }
            sum += intra;
        }
        const bool allOk = (__ballot(!ok) == 0ull);
        if(lane == 0) {
            if(!allOk) { raiseErrorFlag(errorFlag); sum = 0xFFFFFFFFu; }
            *shOffset = sum;
        }
    }
    __syncthreads();
    return *shOffset;
}

// ------------------------------------------------------------------------------------------------
// Ordered append of the flagged neurons of a population to a queue, for spike-like events: the scheme the neuron
// update uses for true spikes (ballot rank in the wave, LDS scan in the block, look-back over per-block counts tagged
// with the step, blocks in groups of 64 with a published group total), as a function every block of the population
// calls with all its threads.  `counts` and `groupTotals` hold one entry per (batch, neuron block of the launch).
// ------------------------------------------------------------------------------------------------
template<bool DIRECT = true>
__device__ __forceinline__ void appendOrdered(bool flag, uint32_t id, uint32_t localBlock, uint32_t numBlocks, size_t aggBase,
                                              unsigned long long *counts, unsigned long long *groupTotals, uint32_t tag,
                                              uint32_t *queue, uint32_t *queueCount, uint32_t *errorFlag,
                                              uint32_t *recordWords = nullptr, bool inRange = false)
{
    __shared__ uint32_t shCount[BLOCK / WAVE];
    __shared__ uint32_t shOffset;
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t wave = threadIdx.x / WAVE;
    const unsigned long long ballot = __ballot(flag);
    // recording: the ballot is the bitfield of this step's events (every word of the step is overwritten)
    if(recordWords && (lane & 31) == 0 && inRange) { recordWords[id >> 5] = (uint32_t)(ballot >> (lane & 32)); }
    const uint32_t laneRank = __popcll(ballot & ((1ull << lane) - 1ull));
    if(lane == 0) { shCount[wave] = __popcll(ballot); }
    __syncthreads();
    uint32_t blockCount = 0, waveOffset = 0;
    #pragma unroll
    for(uint32_t w = 0; w < BLOCK / WAVE; w++) {
        const uint32_t c = shCount[w];
        if(w < wave) { waveOffset += c; }
        blockCount += c;
    }
    const uint32_t prefix = blockQueueOffset<DIRECT>(blockCount, localBlock, numBlocks, aggBase, counts, groupTotals, tag, &shOffset, errorFlag);
    if(prefix != 0xFFFFFFFFu) {
        if(flag) { queue[prefix + waveOffset + laneRank] = id; }
        if(localBlock == numBlocks - 1 && threadIdx.x == 0) { *queueCount = prefix + blockCount; }
    }
    __syncthreads();            // the shared words are reused by the next call
}

// What the populations of a launch may have.  A launch fetches its instructions anew, and a path that jumps over what a population does not have fetches a
// little of each; neuronUpdateKernel is 5,430 and 6,380 instructions (DIRECT) with AnyNeurons, 845 and 1,250 with LeanNeurons.  us a launch, AnyNeurons / LeanNeurons: 4,000 LIF neurons 4.57 / 4.16,
// 17,011 4.92 / 4.52, 100,000 5.72 / 5.44, 300,007 6.02 / 5.68; stepFusedKernel on the microcircuit at 0.35 with Poisson sources, AnyNeurons / RingNeurons 6.60 / 6.00.
// OWN: the path reads what it needs of the descriptor at once and its inputs without a branch, instead of a dozen trips to the scalar cache in between: 17,011
// neurons 4.52 -> 4.27, the others no change.
// The lines, us a step of two launches / of one: LeanNeurons for eight inputs costs networks with two of them, 17,011 neurons 7.4 -> 7.5, 300,007 11.8 -> 13.0 (and what has five 17,011 8.3 -> 7.6,
// 200,000 11.2 -> 12.2), for four sources 11.8 -> 12.4 (two constant currents, 17,011 8.1 -> 7.4); RingNeurons for four inputs 77,000 neurons with Poisson sources 8.2 -> 8.4 (three inputs
// 8.4 -> 8.3, 27,000 6.8 -> 6.5), for four sources nothing (two sources 10,007 6.2 -> 6.0, 50,021 7.5 -> 7.2, 77,000 the same).
struct AnyNeurons       // whatever a description can say
{
    static constexpr uint32_t PSM = GENNMI_MAX_PSM, CS = GENNMI_MAX_CS;
    static constexpr bool RINGS = true, SOURCES = true, SHADOW = true, REST = true, OWN = false;     // dendritic delays; sources other than DC; shadow queues and zero delays; events, presynaptic output, axonal delays
};
struct LeanNeurons      // few inputs without delays, at most a constant current
{
    static constexpr uint32_t PSM = 4, CS = 1;
    static constexpr bool RINGS = false, SOURCES = false, SHADOW = false, REST = false, OWN = true;
};
struct RingNeurons      // the single-launch step's
{
    static constexpr uint32_t PSM = 2, CS = 1;
    static constexpr bool RINGS = true, SOURCES = true, SHADOW = true, REST = false, OWN = false;
};
template<typename HAS>
inline bool neuronsFit(const std::vector<NeuronGroupDev> &groups)
{
    return std::all_of(groups.begin(), groups.end(), [](const NeuronGroupDev &n) {
        const gennmi_neuron_update_group_t &g = n.g;
        bool fits = g.numPSM <= HAS::PSM && g.numCS <= HAS::CS && (HAS::SHADOW || (!n.zeroStart && !n.shadowSpk))
                    && (HAS::REST || (g.numPreOutput == 0 && g.numSpkEvent == 0 && g.numDelaySlots <= 1));
        for(uint32_t m = 0; m < g.numPSM; m++) { fits = fits && (HAS::RINGS || g.psm[m].maxDenDelay == 0); }
        for(uint32_t c = 0; c < g.numCS; c++) { fits = fits && (HAS::SOURCES || g.cs[c].kind == GENNMI_CS_DC); }
        return fits;
    });
}

// ------------------------------------------------------------------------------------------------
// Neuron update.  One lane per neuron.  Spikes are emitted in ascending neuron index (the CPU
// backend's order, single_threaded_cpu/backend.cc:321, 2119-2133): wave ballot gives the in-wave
// rank, an LDS scan the in-block rank, and a look-back over per-block counts published in `agg`
// (tagged with the step so nothing ever needs clearing) the cross-block offset.  Only blocks that
// emitted spikes, and the last block of each population (which stores spkCnt), look back.
// ------------------------------------------------------------------------------------------------
template<typename HAS, bool DIRECT = true>
__device__ __forceinline__ void neuronBody(const NeuronGroupDev &descriptor, uint32_t blockInKernel, uint32_t totalNeuronBlocks,
                                           const StepArgs &st, float dt, unsigned long long *agg, uint32_t *errorFlag)
{
    __shared__ uint32_t shWaveCount[BLOCK / WAVE];
    __shared__ uint32_t shPrefix;

    // (OWN: what the path needs of the descriptor is read at its beginning, at once, instead of where it is needed)
    typename std::conditional<HAS::OWN, const NeuronGroupDev, const NeuronGroupDev&>::type G = descriptor;
    const gennmi_neuron_update_group_t &g = G.g;
    const uint32_t batch = blockIdx.y;
    const uint32_t localBlock = blockInKernel - G.startBlock;
    const uint32_t n = g.numNeurons;
    const uint32_t i = localBlock * BLOCK + threadIdx.x;
    // (a lane beyond the population reads its last neuron and keeps nothing of it)
    const bool present = (i < n);
    const size_t bi = (size_t)batch * n + (HAS::OWN ? min(i, n - 1) : i);
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t wave = threadIdx.x / WAVE;
    const float t = st.t;
    constexpr uint32_t MAX_PSM = HAS::PSM, MAX_CS = HAS::CS;

    bool spiked = false;
    float vEvent = 0.0f;
    uint32_t z0 = 0, z1 = 0;
    if(HAS::SHADOW && G.zeroStart && i < n) { z0 = asGlobal(G.zeroStart)[i]; z1 = asGlobal(G.zeroStart)[i + 1]; }
    // what the update leaves to be stored (see storeState below)
    float l0 = 0, l1 = 0, preTrace = 0, postTrace = 0;
    float lin[MAX_PSM];
    uint32_t ringSlot[MAX_PSM];
    #pragma unroll
    for(uint32_t m = 0; m < MAX_PSM; m++) { lin[m] = 0.0f; }
    if(HAS::OWN || present) {
        // order of operations: neuronUpdateGroupMerged.cc:552-773 — PSMs, current sources, sim code,
        // WU pre/post dynamics, threshold, then (on a spike) WU pre/post spike code, sT, reset
        float nextTime = 0.0f;
        if(g.model == GENNMI_NEURON_SPIKE_SOURCE_ARRAY) {
            // one coalesced read instead of startSpike, endSpike and a gather from spikeTimes: the time of the neuron's next
            // spike is kept beside the state and refreshed only when the neuron fires
            nextTime = asGlobal(G.nextSpikeTime)[bi];
        }
        else {
            // Every load of this neuron's inputs is issued before the first store: the pointers come out of a
            // descriptor in memory, so a store in between would force the compiler to re-read the descriptor
            // and would serialise the loads, and each dependent access costs about a microsecond at the start of
            // a launch (nothing is cached yet).  Sums keep the reference's order (PSMs, then current sources).
            float front[MAX_PSM], inj[MAX_CS], rev[GENNMI_MAX_PRE_OUTPUT];
            const uint32_t numPSM = g.numPSM, numCS = g.numCS, numRev = HAS::REST ? g.numPreOutput : 0u;
            #pragma unroll
            for(uint32_t q = 0; q < GENNMI_MAX_PRE_OUTPUT; q++) { rev[q] = (q < numRev) ? asGlobal(g.outPre[q])[bi] : 0.0f; }
            l0 = asGlobal(g.var0)[bi]; l1 = asGlobal(g.var1)[bi];
            #pragma unroll
            for(uint32_t m = 0; m < MAX_PSM; m++) {
                lin[m] = 0.0f; front[m] = 0.0f;
                if(m < numPSM) {
                    lin[m] = asGlobal(g.psm[m].outPost)[bi];
                    const uint32_t D = HAS::RINGS ? g.psm[m].maxDenDelay : 0u;
                    if(D) {
                        ringSlot[m] = modStep(st.epoch + 1, D);
                        front[m] = asGlobal(g.psm[m].denDelay)[((size_t)batch * D + ringSlot[m]) * n + i];
                    }
                }
            }
            #pragma unroll
            for(uint32_t c = 0; c < MAX_CS; c++) {
                inj[c] = 0.0f;
                if(c < numCS) {
                    inj[c] = (!HAS::SOURCES || g.cs[c].kind == GENNMI_CS_DC) ? g.cs[c].amp
                           : (g.cs[c].kind == GENNMI_CS_ARRAY) ? asGlobal(g.cs[c].array)[(size_t)modStep(st.epoch, g.cs[c].arraySteps) * n + i]
                                                               : poissonExpInject(g.cs[c], asGlobal(g.cs[c].current), bi, st.epoch);
                }
            }
            float Isyn = 0;
            #pragma unroll
            for(uint32_t m = 0; m < MAX_PSM; m++) {
                if(m < numPSM) {
                    // read and clear the front slot of the ring (neuronUpdateGroupMerged.cc:84-101)
                    float linSyn = lin[m];
                    const uint32_t D = HAS::RINGS ? g.psm[m].maxDenDelay : 0u;
                    if(D) { linSyn += front[m]; }
                    if(g.psm[m].kind == GENNMI_PSM_EXPCURR) {
                        Isyn += g.psm[m].init * linSyn;
                        linSyn *= g.psm[m].expDecay;
                    }
                    else {
                        Isyn += linSyn;
                        linSyn = 0.0f;
                    }
                    lin[m] = linSyn;
                }
            }
            // presynaptic output of the outgoing projections: after the postsynaptic models, before the current sources
            #pragma unroll
            for(uint32_t q = 0; q < GENNMI_MAX_PRE_OUTPUT; q++) { if(q < numRev) { Isyn += rev[q]; } }
            #pragma unroll
            for(uint32_t c = 0; c < MAX_CS; c++) { if(c < numCS) { Isyn += inj[c]; } }
            if(g.model == GENNMI_NEURON_LIF) {
                if(l1 <= 0.0f) {
                    const float alpha = ((Isyn + g.params[0]) * g.params[1]) + g.params[2];
                    l0 = alpha - (g.params[3] * (alpha - l0));
                }
                else {
                    l1 -= dt;
                }
            }
            else {
                if(l0 >= 30.0f) {
                    l0 = g.params[2];
                    l1 += g.params[3];
                }
                l0 += 0.5f * (0.04f * l0 * l0 + 5.0f * l0 + 140.0f - l1 + Isyn) * dt;
                l0 += 0.5f * (0.04f * l0 * l0 + 5.0f * l0 + 140.0f - l1 + Isyn) * dt;
                l1 += g.params[0] * (g.params[1] * l0 - l1) * dt;
                if(l0 > 30.0f) { l0 = 30.0f; }
            }
        }
        if(g.preTrace) { preTrace = g.preTrace[bi] * g.preDecay; }
        if(g.postTrace) { postTrace = g.postTrace[bi] * g.postDecay; }
        if(g.model == GENNMI_NEURON_LIF) { spiked = (l1 <= 0.0f && l0 >= g.params[4]); }
        else if(g.model == GENNMI_NEURON_IZHIKEVICH) { spiked = (l0 >= 29.99f); }
        else { spiked = (t >= nextTime); }       // startSpike != endSpike && t >= spikeTimes[startSpike] (neuronModels.h:274-286)
        spiked = spiked && present;
        vEvent = l0;           // spike-like event conditions see the updated V before any reset (neuronUpdateGroupMerged.cc:677-683)
        if(spiked) {
            preTrace += 1.0f; postTrace += 1.0f;
            if(g.model == GENNMI_NEURON_LIF) { l0 = g.params[5]; l1 = g.params[6]; }
        }
    }
    // The stores of the update, issued once the block's spike count is on its way (the work-groups behind this one wait for
    // that count; a wavefront queued behind the chip's store traffic before it can vote would keep them waiting).
    auto storeState = [&]() {
        if(i < n) {
            if(g.model == GENNMI_NEURON_SPIKE_SOURCE_ARRAY) {
                if(spiked) {
                    const uint32_t startSpike = g.startSpike[bi] + 1;
                    g.startSpike[bi] = startSpike;
                    G.nextSpikeTime[bi] = (startSpike != g.endSpike[bi]) ? g.spikeTimes[startSpike] : INFINITY;
                }
            }
            else {
                const uint32_t numPSM = g.numPSM, numRev = HAS::REST ? g.numPreOutput : 0u;
                #pragma unroll
                for(uint32_t q = 0; q < GENNMI_MAX_PRE_OUTPUT; q++) { if(q < numRev) { storeThrough(&asGlobal(g.outPre[q])[bi], 0.0f); } }
                #pragma unroll
                for(uint32_t m = 0; m < MAX_PSM; m++) {
                    if(m < numPSM) {
                        const uint32_t D = HAS::RINGS ? g.psm[m].maxDenDelay : 0u;
                        if(D) { storeThrough(&asGlobal(g.psm[m].denDelay)[((size_t)batch * D + ringSlot[m]) * n + i], 0.0f); }
                        storeThrough(&asGlobal(g.psm[m].outPost)[bi], lin[m]);
                    }
                }
                storeThrough(&asGlobal(g.var0)[bi], l0); storeThrough(&asGlobal(g.var1)[bi], l1);
            }
            if(spiked && g.sT) { g.sT[bi] = t; }
            if(g.preTrace) { storeThrough(&asGlobal(g.preTrace)[bi], preTrace); }
            if(g.postTrace) { storeThrough(&asGlobal(g.postTrace)[bi], postTrace); }
        }
        // keep the user-visible ring pointers current (nothing in the kernels reads them)
        if(HAS::RINGS && localBlock == 0 && batch == 0 && threadIdx.x < g.numPSM) {
            const gennmi_psm_t &psm = g.psm[threadIdx.x];
            if(psm.maxDenDelay && psm.denDelayPtr) { *psm.denDelayPtr = modStep(st.epoch + 1, psm.maxDenDelay); }
        }
    };

    // ---- spike-like events: one ordered queue per event condition ----------------------------------
    if(HAS::REST && g.numSpkEvent) {
        const size_t perArea = (size_t)totalNeuronBlocks * gridDim.y;
        for(uint32_t e = 0; e < g.numSpkEvent; e++) {
            unsigned long long *counts = G.aggEvent + (size_t)e * 2 * perArea;
            appendOrdered<DIRECT>(i < n && vEvent > g.spkEvent[e].threshold, i, localBlock, G.numBlocks, (size_t)batch * totalNeuronBlocks + G.startBlock,
                          counts, counts + perArea, (uint32_t)(st.epoch + 1), g.spkEvent[e].spkEvent + (size_t)batch * n,
                          g.spkEvent[e].spkCntEvent + batch, errorFlag,
                          g.spkEvent[e].recordSpkEvent ? g.spkEvent[e].recordSpkEvent + ((size_t)st.recordingTimestep * gridDim.y + batch) * ((n + 31) / 32) : nullptr, i < n);
        }
    }

    // ---- ordered compaction --------------------------------------------------------------------
    const unsigned long long ballot = __ballot(spiked);
    const uint32_t waveCount = __popcll(ballot);
    const uint32_t laneRank = __popcll(ballot & ((1ull << lane) - 1ull));
    if(lane == 0) { shWaveCount[wave] = waveCount; }

    // recording: the ballot IS the bitfield (bit i%32 of word i/32, runtime.cc:855-913); every word of
    // the step is overwritten, so no clearing and no atomicOr (cf. backendSIMT.cc:1948-1953)
    if(g.recordSpk && (lane & 31) == 0 && i < n) {
        const uint32_t words = (n + 31) / 32;
        g.recordSpk[((size_t)st.recordingTimestep * gridDim.y + batch) * words + (i >> 5)] = (uint32_t)(ballot >> (lane & 32));
    }
    if(G.spikeBitmap && (lane & 31) == 0 && i < n) { G.spikeBitmap[((st.epoch + 1) & 1) * G.bitmapStride + (size_t)batch * ((n + 31) / 32) + (i >> 5)] = (uint32_t)(ballot >> (lane & 32)); }
    __syncthreads();

    uint32_t blockCount = 0, waveOffset = 0;
    #pragma unroll
    for(uint32_t w = 0; w < BLOCK / WAVE; w++) {
        const uint32_t c = shWaveCount[w];
        if(w < wave) { waveOffset += c; }
        blockCount += c;
    }

    const uint32_t tag = (uint32_t)(st.epoch + 1);
    const size_t aggBase = (size_t)batch * totalNeuronBlocks + G.startBlock;
    if(threadIdx.x == 0) {
        // the count itself is all that is communicated, so a relaxed device-scope store suffices
        // (release would write back the whole L2 from every block)
        __hip_atomic_store(&agg[aggBase + localBlock], ((unsigned long long)tag << 32) | blockCount,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    storeState();
    const bool last = (localBlock == G.numBlocks - 1);
    const bool direct = DIRECT && queueDirect(G.numBlocks), groupLeader = (!direct && (localBlock % WAVE) == WAVE - 1) || last;
    if(blockCount == 0 && !groupLeader) { return; }

    // Synapses with d % D == 0 of the neurons that just fired belong in the slot their targets read in the
    // NEXT step, (epoch + 2) % D, which nothing reads or clears during this step — so the presynaptic update of
    // the next step (which skips them) may run concurrently with that step's neuron update.  The wavefront
    // delivers them cooperatively, one fired neuron at a time, lanes striding over its merged list.
    auto deliverZeroDelay = [&]() {
        unsigned long long pending = ballot;
        while(pending) {
            const int src = __ffsll((long long)pending) - 1;
            pending &= pending - 1;
            const uint32_t s0 = __shfl(z0, src, WAVE), s1 = __shfl(z1, src, WAVE);
            for(uint32_t k = s0 + lane; k < s1; k += WAVE) {
                const ZeroDelayEntry e = G.zeroEntries[k];
                const uint32_t slot = modStep(st.epoch + 2, e.maxDenDelay);
                atomicAddF32(asGlobal(e.ringElem) + ((size_t)batch * e.maxDenDelay + slot) * e.numTrgNeurons, *asGlobal(e.weight));
            }
        }
    };
    if(HAS::SHADOW && G.zeroStart && wave != 0) { deliverZeroDelay(); }

    if(!direct && wave == 0) {
        // Two-level offset: blocks of a population form groups of 64.  The last block of a group sums the
        // group's 64 counts and publishes the group total in the second half of `agg`; a block's offset is the
        // sum of the counts of the earlier blocks of its group plus the totals of the earlier groups.  Every
        // wait is for a value that depends only on other blocks having published their own count, so there is
        // no chain of blocks waiting for each other's results, whatever the population size.
        unsigned long long *groupAgg = agg + (size_t)totalNeuronBlocks * gridDim.y;
        const uint32_t group = localBlock / WAVE, inGroup = localBlock % WAVE;
        const size_t groupBase = aggBase + (size_t)group * WAVE;
        bool ok = true;
        auto waitFor = [&](const unsigned long long *p) -> uint32_t {
            uint32_t spins = 0;
            while(true) {
                const unsigned long long a = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if((uint32_t)(a >> 32) == tag) { return (uint32_t)a; }
                if(++spins > c_spinLimit) { ok = false; return 0u; }
                __builtin_amdgcn_s_sleep(1);
            }
        };
        // counts of the earlier blocks of this group (lane == inGroup contributes this block's own count)
        uint32_t v = 0;
        if(lane < inGroup) { v = waitFor(&agg[groupBase + lane]); }
        uint32_t intra = v;
        for(int off = WAVE / 2; off > 0; off >>= 1) { intra += __shfl_down(intra, off, WAVE); }
        intra = __shfl(intra, 0, WAVE);
        if(inGroup == WAVE - 1 || last) {
            if(lane == 0 && ok) {
                __hip_atomic_store(&groupAgg[aggBase + group], ((unsigned long long)tag << 32) | (intra + blockCount),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        uint32_t sum = 0;
        if(blockCount != 0 || last) {
            for(uint32_t base = 0; base < group; base += WAVE) {
                if(base + lane < group) { sum += waitFor(&groupAgg[aggBase + base + lane]); }
            }
            for(int off = WAVE / 2; off > 0; off >>= 1) { sum += __shfl_down(sum, off, WAVE); }
            sum += intra;
        }
        const bool allOk = (__ballot(!ok) == 0ull);
        if(lane == 0) {
            if(!allOk) { raiseErrorFlag(errorFlag); sum = 0xFFFFFFFFu; }
            shPrefix = sum;
        }
    }
    if(!direct) { __syncthreads(); }
    const uint32_t prefix = direct ? sumOfEarlierBlocks(localBlock, agg + aggBase, tag, errorFlag) : shPrefix;
    if(prefix == 0xFFFFFFFFu) { return; }       // bounded wait expired: flagged, nothing written
    // with axonal delay the queue is a ring of slots and this step writes slot (epoch + 1) % slots: the reference's
    // spkQuePtr after the increment at the start of its updateNeurons (neuronUpdateGroupMerged.cc:947-953)
    const uint32_t delaySlots = HAS::REST ? max(1u, g.numDelaySlots) : 1u;
    const size_t queue = (size_t)batch * delaySlots + ((delaySlots > 1) ? modStep(st.epoch + 1, delaySlots) : 0u);
    if(spiked) { g.spk[queue * n + prefix + waveOffset + laneRank] = i; }
    if(last && threadIdx.x == 0) { g.spkCnt[queue] = prefix + blockCount; }
    // further copies of the queue (one population can feed several spike arrays: its own outgoing projections
    // and, for learnPost, the incoming plastic ones; runtime.cc:267-278)
    #pragma unroll
    for(uint32_t q = 0; q < GENNMI_MAX_EXTRA_SPK; q++) {
        if(q < g.numExtraSpk) {
            if(spiked) { g.extraSpk[q][(size_t)batch * n + prefix + waveOffset + laneRank] = i; }
            if(last && threadIdx.x == 0) { g.extraSpkCnt[q][batch] = prefix + blockCount; }
        }
    }
    if(HAS::SHADOW && G.shadowSpk) {
        const uint32_t parity = (uint32_t)(st.epoch & 1);
        if(spiked) { G.shadowSpk[((size_t)parity * gridDim.y + batch) * n + prefix + waveOffset + laneRank] = i; }
        if(last && threadIdx.x == 0) { G.shadowCnt[(size_t)parity * gridDim.y + batch] = prefix + blockCount; }
    }
    if(HAS::SHADOW && G.zeroStart && wave == 0) { deliverZeroDelay(); }
}

// (DIRECT: one of the populations is queueDirect.  Where none is, a step that has that code compiled in is slower: DENSE 8192 x 8192 stepped 9.75 us a step
// before there was such code, 9.91 with it, 9.79 without; 1000 x 500 batch 4 8.85, 9.02 and 8.88)
template<typename HAS, bool DIRECT>
__global__ __launch_bounds__(BLOCK)
void neuronUpdateKernel(const NeuronGroupDev * __restrict__ blocks, StepArgs args, float dt,
                        unsigned long long *agg, uint32_t *errorFlag)
{
    neuronBody<HAS, DIRECT>(blocks[blockIdx.x], blockIdx.x, gridDim.x, args, dt, agg, errorFlag);
}

// ------------------------------------------------------------------------------------------------
// Neuron update for large populations.  With one neuron per lane a population of millions is many rounds of resident
// work-groups, and every round pays the whole dependent chain (descriptor, inputs, count published, look-back, queue).
// Here a wavefront takes NPL consecutive chunks of 64 neurons: all inputs of all chunks are requested before anything is
// stored, so a lane has NPL times the bytes in flight and the launch has 1/NPL of the work-groups.  Same arithmetic per
// neuron and the same ordered queue as neuronBody (chunks of a wave are consecutive neurons, so chunk-major rank is neuron
// order); the subset of features large populations use: LIF, Izhikevich and spike-source groups with up to two
// postsynaptic models and one current source, spike recording; no traces, spike times, delay slots, further spike arrays,
// events or presynaptic output (the host picks this kernel only when every group fits).
// ------------------------------------------------------------------------------------------------
constexpr uint32_t BULK_MAX_PSM = 2, BULK_MAX_CS = 1;

// What the update of a plain neuron needs of its group, read once into registers: the descriptor lives in global memory, and
// behind every store the compiler would read its fields again (a store may alias anything), ten dependent scalar loads per neuron.
struct PlainNeuron
{
    uint32_t model;
    float p[7];
};
__device__ __forceinline__ PlainNeuron plainNeuronOf(const gennmi_neuron_update_group_t &g)
{
    PlainNeuron c;
    c.model = g.model;
    #pragma unroll
    for(int k = 0; k < 7; k++) { c.p[k] = g.params[k]; }
    return c;
}
// sim code, threshold and reset of a LIF (neuronModels.h:220-257) or Izhikevich (:163-186) neuron from its summed input:
// operations and their order as in neuronBody
__device__ __forceinline__ bool plainNeuronStep(const PlainNeuron &c, float Isyn, float dt, float &v0, float &v1)
{
    bool spiked;
    if(c.model == GENNMI_NEURON_LIF) {
        if(v1 <= 0.0f) {
            const float alpha = ((Isyn + c.p[0]) * c.p[1]) + c.p[2];
            v0 = alpha - (c.p[3] * (alpha - v0));
        }
        else {
            v1 -= dt;
        }
        spiked = (v1 <= 0.0f && v0 >= c.p[4]);
        if(spiked) { v0 = c.p[5]; v1 = c.p[6]; }
    }
    else {
        if(v0 >= 30.0f) {
            v0 = c.p[2];
            v1 += c.p[3];
        }
        v0 += 0.5f * (0.04f * v0 * v0 + 5.0f * v0 + 140.0f - v1 + Isyn) * dt;
        v0 += 0.5f * (0.04f * v0 * v0 + 5.0f * v0 + 140.0f - v1 + Isyn) * dt;
        v1 += c.p[0] * (c.p[1] * v0 - v1) * dt;
        if(v0 > 30.0f) { v0 = 30.0f; }
        spiked = (v0 >= 29.99f);
    }
    return spiked;
}

// (THREADS: threads of the calling work-group, all of which call; batch / numBatches: the grid's second dimension in the neuron kernels)
// (LEAN: no population is a spike source or has dendritic delays; see AnyNeurons.  1,660 instructions for four chunks instead of 2,690, and of 5,890 while what is
// uniform was decided chunk by chunk: 10^6 Izhikevich neurons 8.8 -> 7.8 us a launch with LEAN alone, 6.8 with straight loads and one decision besides)
// (STRAIGHT: a chunk's spiking sources are looked up without a branch, so that a lane's chunks do not wait for one another: a step of a convolution 64x64x16 -> 32,
// batch 16, whose neurons have a kernel of their own, 38.6 us -> 31.3 with eight chunks, 30.3 -> 29.4 with four, 37.2 -> 36.2 with two; 1.4 x 10^6 neurons with delays, eight chunks,
// 25.8 -> 22.4.  The convolution's one-launch step, whose other work-groups wait for memory as well, is slower with it: 28.3 -> 29.4)
template<int NPL, int THREADS = BLOCK, bool DIRECT = true, bool LEAN = false, bool STRAIGHT = false>
__device__ __forceinline__ void neuronBulkBody(const NeuronGroupDev &G, uint32_t blockInKernel, uint32_t totalNeuronBlocks,
                                               const StepArgs &st, float dt, unsigned long long *agg, uint32_t *errorFlag,
                                               uint32_t batch, uint32_t numBatches)
{
    __shared__ uint32_t shWaveCount[THREADS / WAVE];
    __shared__ uint32_t shPrefix;
    const gennmi_neuron_update_group_t &g = G.g;
    const uint32_t localBlock = blockInKernel - G.startBlock;
    const uint32_t n = g.numNeurons;
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t wave = threadIdx.x / WAVE;
    const float t = st.t;
    const uint32_t first = (localBlock * (THREADS / WAVE) + wave) * (WAVE * NPL) + lane;      // this lane's neuron in chunk 0
    const uint32_t numPSM = g.numPSM, numCS = g.numCS;
    // the group's constants and array addresses, read once (see PlainNeuron)
    const PlainNeuron constants = plainNeuronOf(g);
    const bool source = !LEAN && (constants.model == GENNMI_NEURON_SPIKE_SOURCE_ARRAY);
    GLOBAL_AS float *var0 = asGlobal(g.var0), *var1 = asGlobal(g.var1);
    GLOBAL_AS float *psmOut[BULK_MAX_PSM], *psmRing[BULK_MAX_PSM];
    uint32_t psmD[BULK_MAX_PSM], psmKind[BULK_MAX_PSM];
    float psmInit[BULK_MAX_PSM], psmDecay[BULK_MAX_PSM];
    #pragma unroll
    for(uint32_t m = 0; m < BULK_MAX_PSM; m++) {
        const bool have = (m < numPSM);
        psmOut[m] = have ? asGlobal(g.psm[m].outPost) : nullptr; psmRing[m] = have ? asGlobal(g.psm[m].denDelay) : nullptr;
        psmD[m] = (!LEAN && have) ? g.psm[m].maxDenDelay : 0u; psmKind[m] = have ? g.psm[m].kind : 0u;
        psmInit[m] = have ? g.psm[m].init : 0.0f; psmDecay[m] = have ? g.psm[m].expDecay : 0.0f;
    }
    uint32_t ringSlot[BULK_MAX_PSM];
    #pragma unroll
    for(uint32_t m = 0; m < BULK_MAX_PSM; m++) { ringSlot[m] = psmD[m] ? modStep(st.epoch + 1, psmD[m]) : 0u; }
    const uint32_t csKind = numCS ? g.cs[0].kind : 0u, csRow = (numCS && csKind == GENNMI_CS_ARRAY) ? modStep(st.epoch, g.cs[0].arraySteps) : 0u;
    const float csAmp = numCS ? g.cs[0].amp : 0.0f;
    GLOBAL_AS const float *csArray = numCS ? asGlobal(g.cs[0].array) : nullptr;
    uint32_t *recordSpk = g.recordSpk, *spikeBitmap = G.spikeBitmap;
    uint32_t *startSpikeArr = g.startSpike; const uint32_t *endSpikeArr = g.endSpike; const float *spikeTimesArr = g.spikeTimes;
    float *nextSpikeTime = G.nextSpikeTime;
    const size_t bitmapStride = G.bitmapStride;
    uint32_t *spkQueue = g.spk, *spkCount = g.spkCnt;
    const uint32_t groupBlocks = G.numBlocks, groupStart = G.startBlock;

    float l0[NPL], l1[NPL], lin[NPL][BULK_MAX_PSM], front[NPL][BULK_MAX_PSM], inj[NPL];
    bool spiked[NPL];
    // ---- every input of every chunk first.  What is uniform is decided once for all chunks, so that a launch runs through few instructions (see AnyNeurons); a
    // lane beyond the population reads its last neuron and keeps nothing of it.
    uint32_t ids[NPL];
    #pragma unroll
    for(int j = 0; j < NPL; j++) {
        ids[j] = min(first + j * WAVE, n - 1);
        l0[j] = l1[j] = inj[j] = 0.0f;
        #pragma unroll
        for(uint32_t m = 0; m < BULK_MAX_PSM; m++) { lin[j][m] = front[j][m] = 0.0f; }
    }
    const size_t batchBase = (size_t)batch * n;
    if(source) {
        #pragma unroll
        for(int j = 0; j < NPL; j++) { l0[j] = asGlobal(nextSpikeTime)[batchBase + ids[j]]; }
    }
    else {
        #pragma unroll
        for(int j = 0; j < NPL; j++) { l0[j] = var0[batchBase + ids[j]]; l1[j] = var1[batchBase + ids[j]]; }
        #pragma unroll
        for(uint32_t m = 0; m < BULK_MAX_PSM; m++) {
            if(m < numPSM) {
                #pragma unroll
                for(int j = 0; j < NPL; j++) { lin[j][m] = psmOut[m][batchBase + ids[j]]; }
                const uint32_t D = psmD[m];
                if(D) {
                    GLOBAL_AS const float *slot = psmRing[m] + ((size_t)batch * D + ringSlot[m]) * n;
                    #pragma unroll
                    for(int j = 0; j < NPL; j++) { front[j][m] = slot[ids[j]]; }
                }
            }
        }
        if(csKind == GENNMI_CS_ARRAY && numCS) {
            GLOBAL_AS const float *row = csArray + (size_t)csRow * n;
            #pragma unroll
            for(int j = 0; j < NPL; j++) { inj[j] = row[ids[j]]; }
        }
        else {
            #pragma unroll
            for(int j = 0; j < NPL; j++) { inj[j] = csAmp; }
        }
    }
    // ---- update, chunk by chunk (operations and their order as in neuronBody); results stay in registers until the block's
    // spike count is on its way: work-groups behind this one wait for that count, and a wavefront that has to queue
    // behind the store traffic of the whole chip before it can vote would keep them waiting
    float outLin[NPL][BULK_MAX_PSM];
    uint32_t newStart[NPL];
    auto update = [&](auto model) {
        PlainNeuron neuron = constants;
        neuron.model = model.value;
        #pragma unroll
        for(int j = 0; j < NPL; j++) {
            float Isyn = 0;
            #pragma unroll
            for(uint32_t m = 0; m < BULK_MAX_PSM; m++) {
                outLin[j][m] = 0.0f;
                if(m < numPSM) {
                    float linSyn = lin[j][m];
                    const uint32_t D = psmD[m];
                    if(D) { linSyn += front[j][m]; }
                    const bool exponential = (psmKind[m] == GENNMI_PSM_EXPCURR);
                    Isyn += exponential ? psmInit[m] * linSyn : linSyn;
                    outLin[j][m] = exponential ? linSyn * psmDecay[m] : 0.0f;
                }
            }
            if(numCS) { Isyn += inj[j]; }
            spiked[j] = plainNeuronStep(neuron, Isyn, dt, l0[j], l1[j]) && first + j * WAVE < n;
        }
    };
    if(source) {
        #pragma unroll
        for(int j = 0; j < NPL; j++) {
            spiked[j] = (t >= l0[j]) && first + j * WAVE < n;
            if(STRAIGHT) { newStart[j] = asGlobal(startSpikeArr)[batchBase + (spiked[j] ? ids[j] : ids[0])] + 1; }
            else { newStart[j] = spiked[j] ? startSpikeArr[batchBase + ids[j]] + 1 : 0u; }
        }
    }
    else if(constants.model == GENNMI_NEURON_LIF) { update(std::integral_constant<uint32_t, GENNMI_NEURON_LIF>()); }
    else { update(std::integral_constant<uint32_t, GENNMI_NEURON_IZHIKEVICH>()); }

    // ---- ordered compaction: rank = spikes of the wave's earlier chunks + spikes of lower lanes in this chunk
    uint32_t rank[NPL];
    unsigned long long ballots[NPL];
    uint32_t waveCount = 0;
    #pragma unroll
    for(int j = 0; j < NPL; j++) {
        ballots[j] = __ballot(spiked[j]);
        rank[j] = waveCount + __popcll(ballots[j] & ((1ull << lane) - 1ull));
        waveCount += __popcll(ballots[j]);
    }
    if(lane == 0) { shWaveCount[wave] = waveCount; }
    __syncthreads();
    uint32_t blockCount = 0, waveOffset = 0;
    #pragma unroll
    for(uint32_t w = 0; w < THREADS / WAVE; w++) {
        const uint32_t c = shWaveCount[w];
        if(w < wave) { waveOffset += c; }
        blockCount += c;
    }
    unsigned long long *groupAgg = agg + (size_t)totalNeuronBlocks * numBatches;
    const size_t aggBase = (size_t)batch * totalNeuronBlocks + groupStart;
    publishBlockCount(blockCount, localBlock, aggBase, agg, (uint32_t)(st.epoch + 1));

    // ---- state, recording words and bitmap
    #pragma unroll
    for(int j = 0; j < NPL; j++) {
        const uint32_t i = first + j * WAVE;
        const size_t bi = (size_t)batch * n + i;
        if(i >= n) { continue; }
        if(recordSpk && (lane & 31) == 0) {
            const uint32_t words = (n + 31) / 32;
            recordSpk[((size_t)st.recordingTimestep * numBatches + batch) * words + (i >> 5)] = (uint32_t)(ballots[j] >> (lane & 32));
        }
        if(spikeBitmap && (lane & 31) == 0) { spikeBitmap[((st.epoch + 1) & 1) * bitmapStride + (size_t)batch * ((n + 31) / 32) + (i >> 5)] = (uint32_t)(ballots[j] >> (lane & 32)); }
        if(source) {
            if(spiked[j]) {
                startSpikeArr[bi] = newStart[j];
                nextSpikeTime[bi] = (newStart[j] != endSpikeArr[bi]) ? spikeTimesArr[newStart[j]] : INFINITY;
            }
            continue;
        }
        #pragma unroll
        for(uint32_t m = 0; m < BULK_MAX_PSM; m++) {
            if(m < numPSM) {
                const uint32_t D = psmD[m];
                if(D) { storeThrough(&psmRing[m][((size_t)batch * D + ringSlot[m]) * n + i], 0.0f); }
                // (an input that is the same bits as it was read — a DeltaCurr input that received nothing: zero in, zero out —
                // is not written again: in a quiet step that is most of a population's 4 bytes per neuron)
                if(__float_as_uint(outLin[j][m]) != __float_as_uint(lin[j][m])) { storeThrough(&psmOut[m][bi], outLin[j][m]); }
            }
        }
        storeThrough(&var0[bi], l0[j]); storeThrough(&var1[bi], l1[j]);
    }
    if(!LEAN && localBlock == 0 && batch == 0 && threadIdx.x < g.numPSM) {
        const gennmi_psm_t &psm = g.psm[threadIdx.x];
        if(psm.maxDenDelay && psm.denDelayPtr) { *psm.denDelayPtr = modStep(st.epoch + 1, psm.maxDenDelay); }
    }

    const uint32_t prefix = blockQueueOffset<DIRECT>(blockCount, localBlock, groupBlocks, aggBase, agg, groupAgg,
                                                     (uint32_t)(st.epoch + 1), &shPrefix, errorFlag, true);
    if(prefix == 0xFFFFFFFFu) { return; }
    #pragma unroll
    for(int j = 0; j < NPL; j++) {
        if(spiked[j]) { spkQueue[(size_t)batch * n + prefix + waveOffset + rank[j]] = first + j * WAVE; }
    }
    if(localBlock == groupBlocks - 1 && threadIdx.x == 0) { spkCount[batch] = prefix + blockCount; }
}

template<int NPL, bool LEAN>
__global__ __launch_bounds__(BLOCK)
void neuronBulkKernel(const NeuronGroupDev * __restrict__ blocks, StepArgs args, float dt, unsigned long long *agg, uint32_t *errorFlag)
{
    neuronBulkBody<NPL, BLOCK, true, LEAN, true>(blocks[blockIdx.x], blockIdx.x, gridDim.x, args, dt, agg, errorFlag, blockIdx.y, gridDim.y);
}

// One launch per timestep for networks whose projections all go through the dendritic-delay ring: the
// neuron update of step t and the presynaptic update of step t touch disjoint ring slots once zero-delay
// synapses are delivered by the spiking neuron itself, and the presynaptic update reads the shadow spike
// queue of step t-1 while the neuron update refills the visible one.  Neuron blocks come first so that
// their look-back chain starts early.  (Instances: RingNeurons with DelayRows, and AnyNeurons with AnyRows.  AnyNeurons with DelayRows, 58 registers instead of
// 84, is slower, us a step: 2 x 100 delayed synapses a neuron and two current sources, 10,007 neurons 6.2 -> 6.4, 50,021 7.4 -> 8.0, 77,000 8.4 -> 8.8, 150,001 9.6 both.)
template<typename HAS, typename ROWS>
__global__ __launch_bounds__(BLOCK)
void stepFusedKernel(const NeuronGroupDev * __restrict__ neuronBlocks, uint32_t numNeuronBlocks, const PreGroupDev * __restrict__ preBlocks,
                     StepArgs args, float dt, unsigned long long *agg, uint32_t *errorFlag, unsigned long long *eventCounter)
{
    const StepArgs st = args;
    if(blockIdx.x < numNeuronBlocks) {
        // the neuron blocks are the critical path (other blocks wait for their spike counts): let their
        // instructions issue ahead of the presynaptic blocks that share the compute unit
        __builtin_amdgcn_s_setprio(3);
        // (offsets in two levels throughout: 50 steps of the full microcircuit 562 us, with sumOfEarlierBlocks in this kernel 569.  2000 steps of 0.35 of it
        // 13.50 ms in this kernel before there was a sumOfEarlierBlocks, 13.66 with it for spike-like events only, which no step there has, 13.27 without)
        neuronBody<HAS, false>(neuronBlocks[blockIdx.x], blockIdx.x, numNeuronBlocks, st, dt, agg, errorFlag);
    }
    else { presynapticBody<ROWS>(preBlocks[blockIdx.x - numNeuronBlocks], blockIdx.x - numNeuronBlocks, blockIdx.y, gridDim.y, st, dt, eventCounter); }
}

// Per row: count the synapses with d % D == 0 and, when `entries` is given, append them at offset[row].
__global__ void zeroDelayScanKernel(uint32_t numSrc, uint32_t rowStride, const uint32_t *rowLength, const uint8_t *d, uint32_t D,
                                    const uint32_t *ind, const float *g, float *denDelay, uint32_t numTrg,
                                    uint32_t *zeroLen, const uint32_t *offset, ZeroDelayEntry *entries)
{
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if(row >= numSrc) { return; }
    const size_t base = (size_t)row * rowStride;
    uint32_t count = 0;
    for(uint32_t j = 0; j < rowLength[row]; j++) {
        if((d[base + j] % D) == 0) {
            if(entries) { entries[offset[row] + count] = ZeroDelayEntry{denDelay + ind[base + j], g + base + j, numTrg, D}; }
            count++;
        }
    }
    if(zeroLen) { zeroLen[row] = count; }
}

// spike sources: (re)build the per-neuron copy of the next spike time from the arrays the user owns
__global__ void nextSpikeTimeKernel(const uint32_t *startSpike, const uint32_t *endSpike, const float *spikeTimes, float *next, size_t count)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i < count) {
        const uint32_t s = startSpike[i];
        next[i] = (s != endSpike[i]) ? spikeTimes[s] : INFINITY;
    }
}

// four floats per lane; dwordx4 when both pointers are 16-byte aligned (hipMalloc'd arrays are), else scalar
// early deliveries of zero-delay synapses that have to be added or taken back after the connectivity was rewritten
struct ZeroDelayCorrection { float *target; const float *weight; float sign; uint32_t pad_; };
__global__ void zeroDelayCorrectionKernel(const ZeroDelayCorrection *fix, uint32_t count)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if(k < count) { atomicAddF32(asGlobal(fix[k].target), fix[k].sign * fix[k].weight[0]); }
}

__global__ void copyKernel(float *dst, const float *src, size_t n)
{
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if(i + 4 <= n && ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0) {
        *reinterpret_cast<f32x4*>(dst + i) = *reinterpret_cast<const f32x4*>(src + i);
    }
    else {
        for(size_t k = i; k < n && k < i + 4; k++) { dst[k] = src[k]; }
    }
}

__global__ void fillKernel(float *p, float v, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) { p[i] = v; }
}

}   // namespace

#endif
