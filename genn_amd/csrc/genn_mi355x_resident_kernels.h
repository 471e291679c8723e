// Part of libgenn_mi355x.so: included by genn_mi355x.hip only (one translation unit).
#ifndef GENN_MI355X_RESIDENT_KERNELS_H
#define GENN_MI355X_RESIDENT_KERNELS_H


// ------------------------------------------------------------------------------------------------
// ------------------------------------------------------------------------------------------------
// Resident plan: many timesteps per launch for networks small enough to live on the chip.
//
// A timestep of such a network moves a few megabytes — half a microsecond of HBM time — but as a chain of
// launches it costs ~12 us: ~4 us per kernel boundary (every L2 is written back and invalidated), then step
// state -> spike count -> spike ids -> rows -> ~10^5 scattered fp32 atomics that retire at ~20 G/s on the memory
// side.  Here one work-group owns a tile of neurons for a whole run: their state stays in registers, their
// postsynaptic input (inSyn) and their slice of every dendritic-delay ring stay in LDS, and the only thing
// work-groups exchange is each step's spikes — one 64-bit word per tile (sequence number, count, and up to three
// ids; longer lists go through a side buffer).  Every tile reads the words of
// all tiles, looks up which part of each spiking row targets its own neurons (a per-(row, tile) segment table
// built once; rows are sorted by target), and adds those synapses into its LDS ring: no global atomics, no
// global read-modify-write of the ring, no kernel boundary.  The words are double-buffered by step parity: a
// tile can run at most one step ahead of the slowest one, because it needs every tile's word of step s before
// it can publish its own word of step s+1.
//
// The wait for the other tiles' words is bounded (c_spinLimit polls) and also watches the error flag, so a launch
// whose work-groups are not all resident ends with an error instead of hanging.  Launches of several runners that do not fit on the
// chip together take turns (residentRoom() on the host).
// ------------------------------------------------------------------------------------------------
// Neurons of a tile.  A network takes the smallest of these with which its tiles have a compute unit each: work-groups that share one take twice
// as long around their loop, and every tile waits for the slowest; and with T x T neurons at most each of a tile's T threads has
// one other tile's word to look for.  us a step with tiles of 256, two and four to a compute unit / with these: the full microcircuit 4.4 / 4.1
// (320), 100,000 x 80 5.9 / 5.0 (512), 180,000 x 100 9.0 / 5.7 and 250,000 x 200 10.5 / 4.9 (1024).  Larger ones than needed do not pay: 4,000 x 80
// to 40,000 x 80 within 3 % with 512, up to 20 % more with 1024; the microcircuit at half size 2.8 -> 3.3 with 512.
// Tiles of 320 are for networks with walkers, 65,500 to 82,000 neurons.  us a step with tiles of 256 that share units / 320 / 512: with row parts of eight
// synapses and more the microcircuit with PoissonExp sources at full size - / 4.00 / 5.03 and at 0.86 - / 3.65 / 4.47, 8 x 8,600 neurons x 800 - / 11.8 / 14.0,
// 2 x 40,000 x 1,000 - / 27.3 / 28.1; with a few, 512 would be the better one: 4 x 19,000 x 200 9.7 / 6.2 / 5.4, 4 x 19,000 x 40 6.8 / 4.4 / 3.9,
// 8 x 8,600 x 100 6.1 / 4.4 / 3.9.
// Some networks of many populations have no tile that fits, since every population is rounded up to whole tiles: 40 x 6,200 neurons are 280 tiles of
// 1024.  They step with the other plans, where tiles of 256, four to a unit, once took them: us a step then / now, 80 targets each 11.0 / 11.4, 800 targets 34 / 24.
constexpr uint32_t RES_TILES[] = {256, 320, 512, 1024};
constexpr uint32_t RES_MAX_TILE = 1024;
constexpr uint32_t RES_MAX_PROJ = 16;        // projections into one population
constexpr uint32_t RES_MAX_GROUPS = 64;      // neuron groups
constexpr uint32_t RES_PAIR_CAP = 1024;      // (spike, projection) pairs a tile lists per exchange
// A segment entry says where a row's part inside a tile is and holds its due synapses, those that land in the slot the target reads in the
// very step that delivers them (without a ring all of the part): a step waits for nothing else, and the dependent trip to the records is
// spared.  Entries of a network are of 2, 4 or 8 quads of 16 bytes, which hold 4, 10 or 22 of them; a part with more is walked before the update,
// and every tile waits for the one that does.  us a step of a balanced network, without / with synapses inside entries: 100,000 neurons x
// 80 targets 8.1 / 6.7, 40,000 x 80 4.7 / 4.3 (2 quads), 12,000 x 100 4.19 / 4.00, 4,000 x 80 3.79 / 3.62 (8, which one lane read then), and 2.85 -> 2.47
// since eight lanes read an entry of 8, a quad each; with 2 / with what the host's rule takes now: 4,000 x 80 2.66 / 2.24 (8), 20,000 x 100
// 3.13 / 2.43 and 40,000 x 80 3.52 / 3.26 (4).  Networks with walkers have entries of 4 and no others (the microcircuit, whose rings have few that are
// due, took 4.22 with 2 and with 4), and so have most with PoissonExp sources or more than two postsynaptic models: the host's table of instances.
constexpr uint32_t residentInside(uint32_t quads) { return 3 * quads - 2; }
constexpr uint32_t RES_MAX_QUADS = 8, RES_COUNT_SHIFT = 30;       // a quad's last word: targets, 10 bits each, and the number of its synapses
constexpr uint32_t RES_SEG_OVERFLOW = 1u << 24, RES_SEG_NO_DELAY = 1u << 25;
constexpr uint32_t RES_SEG_PROJ_SHIFT = 26;  // in the kernel's list of pairs: the projection, above an entry's flags
// word: upper half sequence number << 11 | count, lower half up to three tile-local neuron indices, 10 bits each
constexpr uint32_t RES_COUNT_BITS = 11, RES_COUNT_MASK = (1u << RES_COUNT_BITS) - 1u;
constexpr uint32_t RES_SEQ_MASK = (1u << (32 - RES_COUNT_BITS)) - 1u;    // sequence numbers run on from launch to launch, modulo 2^21
constexpr uint32_t RES_WORD_IDS = 3;         // spikes of a tile and step that travel inside its word (more: side buffer)
constexpr uint32_t RES_ID_BITS = 10, RES_ID_MASK = (1u << RES_ID_BITS) - 1u;
constexpr uint32_t RES_REPLICAS = 8;         // copies of the word array, one per XCD, so that polling spreads over memory channels

struct ResProj
{
    const u32x2 *packed;                // one record per (padded) synapse, see residentPackKernel
    const u32x4 *seg;                   // [numSrc * tilesInGroup][QUADS]: the row's part inside a tile, see residentSegKernel
    uint32_t D;                         // ring depth; 0 = no dendritic delay, events add to inSyn
    uint32_t lds;                       // float offset of the ring (D x tile size, slot-major) or inSyn row in the tile's LDS
    uint32_t srcGroup;
    uint32_t pad_[3];
};

struct ResTile
{
    uint32_t group, first, count;       // neuron group, first neuron, neurons in this tile
    uint32_t tileInGroup, tilesInGroup, firstTileOfGroup;
    uint32_t numProj, ldsFloats;
    uint32_t ldsIn[GENNMI_MAX_PSM];     // float offset of the inSyn row of postsynaptic model m
    uint32_t ldsRing[GENNMI_MAX_PSM];   // float offset of its ring (when maxDenDelay > 0)
    ResProj proj[RES_MAX_PROJ];
};

// One entry per (row, tile of the target population).  Its first quad: first idSyn of the row's part inside the tile; its length | number of
// synapses inside << 16 | flags; a weight; targets and count as in every quad's last word.  The others: three weights, targets and count.
// RES_SEG_OVERFLOW: the part has more due synapses than fit (none is inside, the row part is walked before the update);
// RES_SEG_NO_DELAY: the projection has no ring, every synapse is due at once.
__global__ void residentSegKernel(uint32_t numSrc, uint32_t rowStride, const uint32_t *rowLength, const uint32_t *ind, const float *weight,
                                  const uint8_t *delay, uint32_t depth, uint32_t tileSize, uint32_t tilesInGroup, uint32_t quads, u32x4 *seg)
{
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(id >= (size_t)numSrc * tilesInGroup) { return; }
    const uint32_t row = (uint32_t)(id / tilesInGroup), tile = (uint32_t)(id % tilesInGroup);
    const uint32_t len = rowLength[row];
    const uint32_t *r = ind + (size_t)row * rowStride;
    auto lowerBound = [&](uint32_t key) {
        uint32_t lo = 0, hi = len;
        while(lo < hi) { const uint32_t mid = (lo + hi) / 2; if(r[mid] < key) { lo = mid + 1; } else { hi = mid; } }
        return lo;
    };
    const uint32_t a = lowerBound(tile * tileSize), b = lowerBound((tile + 1) * tileSize);
    const uint32_t start = row * rowStride + a;
    uint32_t flags = depth ? 0u : RES_SEG_NO_DELAY;
    auto due = [&](uint32_t j) { return !depth || delay[(size_t)row * rowStride + j] % depth == 0; };
    uint32_t inside = 0;
    for(uint32_t j = a; j < b && inside <= residentInside(quads); j++) { inside += due(j) ? 1u : 0u; }
    if(inside > residentInside(quads)) { flags |= RES_SEG_OVERFLOW; inside = 0; }
    uint32_t j = a, done = 0;
    for(uint32_t q = 0; q < quads; q++) {
        uint32_t x0 = 0, x1 = 0, x2 = 0, last = 0, n = 0;
        if(q == 0) { x0 = start; x1 = min(b - a, 0xFFFFu) | (inside << 16) | flags; }
        for(uint32_t f = q ? 0u : 2u; f < 3 && done < inside; f++, j++, n++, done++) {
            while(!due(j)) { j++; }
            const uint32_t w = __float_as_uint(weight[(size_t)row * rowStride + j]);
            if(f == 0) { x0 = w; } else if(f == 1) { x1 = w; } else { x2 = w; }
            last |= (r[j] - tile * tileSize) << (RES_ID_BITS * n);
        }
        seg[quads * id + q] = u32x4{x0, x1, x2, last | (n << RES_COUNT_SHIFT)};
    }
}

// How many of a sample of a projection's synapses are due: counts[0] of counts[1] (64 rows across the source population, a work-group each)
__global__ __launch_bounds__(BLOCK)
void residentDueKernel(uint32_t numSrc, uint32_t rowStride, const uint32_t *rowLength, const uint8_t *delay, uint32_t depth, uint32_t *counts)
{
    const size_t row = (size_t)blockIdx.x * numSrc / gridDim.x;
    const uint32_t len = rowLength[row];
    uint32_t due = 0;
    for(uint32_t j = threadIdx.x; j < len; j += BLOCK) { due += (delay[row * rowStride + j] % depth == 0) ? 1u : 0u; }
    for(int off = WAVE / 2; off > 0; off >>= 1) { due += __shfl_down(due, off, WAVE); }
    if((threadIdx.x & (WAVE - 1)) == 0 && due) { atomicAdd(&counts[0], due); }
    if(threadIdx.x == 0) { atomicAdd(&counts[1], len); }
}

// The synapses as the row walk reads them: where in the tile's ring they land, in bytes from its front slot (slots of a float a
// neuron of the tile; below the first slot's end: due), and the weight's bits — one 8-byte load per synapse instead of three loads from three arrays (three pages, three cache
// lines per row part), and an addition and a minimum instead of a division by the ring's depth.
// Same index as the arrays it is made from; padding beyond a row's length is copied as it is and never read.
__global__ void residentPackKernel(size_t numSynapses, const uint32_t *ind, const float *weight, const uint8_t *delay, uint32_t depth, uint32_t tileSize, u32x2 *packed)
{
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(id >= numSynapses) { return; }
    u32x2 rec;
    rec.x = 4u * (ind[id] % tileSize + (depth ? ((uint32_t)delay[id] % depth) * tileSize : 0u)); rec.y = __float_as_uint(weight[id]);
    packed[id] = rec;
}

// rows must ascend for the segments to be contiguous
__global__ void residentSortedKernel(uint32_t numSrc, uint32_t rowStride, const uint32_t *rowLength, const uint32_t *ind, uint32_t *unsorted)
{
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(id >= (size_t)numSrc * rowStride) { return; }
    const uint32_t row = (uint32_t)(id / rowStride), j = (uint32_t)(id % rowStride);
    if(j + 1 < rowLength[row] && ind[id] > ind[id + 1]) { *unsorted = 1; }
}

__device__ __forceinline__ uint32_t waveInclusiveScanU32(uint32_t v, uint32_t lane)
{
    #pragma unroll
    for(int d = 1; d < WAVE; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, WAVE);
        if(lane >= (uint32_t)d) { v += o; }
    }
    return v;
}

// Waits for the work-group with its LDS accesses done, and for nothing else: global loads and stores stay in flight.
__device__ __forceinline__ void ldsBarrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The step is a chain of latencies, and what bounds it is the number of links: words arrive -> segment entries -> update -> word.
// The thread that sees a tile's word reads the entries of that tile's spikes itself and adds what is due at once, so there
// is one barrier in a step, between the words and the update (every due synapse is in); the wavefront that finishes the update last
// publishes the tile's word.  The pairs are listed on the side, and the synapses that are not due are added by WALK wavefronts of
// their own, between that barrier and the next one: a step lasts as long as the slowest tile takes around its loop, and time stamps
// showed that tile never waiting for a word, but walking, polling, reading entries and updating one after the other.
// us a step, with five barriers and the walk behind the word / now: the full microcircuit 6.1 / 4.1, with PoissonExp sources at half size
// 5.3 / 2.8, balanced networks of 4,000 x 80 3.8 / 2.85, 100,000 x 80 7.2 / 5.0.  (Spikes taken one after another by the thread that
// watches their word, however many: 180,000 x 100 10.1 -> 15.9.)
// What consecutive exchanges share exists once for each of them: pair lists twice, counters and ring fronts four times (those of the
// exchange after the next are prepared behind the barrier, so no thread meets them half prepared).
// POISSON: some population has a PoissonExp current source (its state then lives in a register per source and neuron);
// the instantiation without it carries neither the registers nor the generator.  QUADS: of a segment entry.
// NPSM: postsynaptic models of any group.  TILE: neurons of a tile, and threads that own one.  WALK: wavefronts beyond those that
// own the tile's neurons; 0: these walk too, once they have published.  With walkers nothing holds a wavefront back between its
// update and the next exchange, so every projection must have a ring of two slots or more: what an early wavefront adds then goes to another slot
// than the one a late one is reading and clearing.  Without, a barrier behind the update keeps them apart, and inSyn itself can be added to.
template<bool POISSON, uint32_t QUADS, uint32_t NPSM, uint32_t TILE, uint32_t WALK>
__global__ __launch_bounds__(TILE + WALK * WAVE, (TILE + WALK * WAVE + 4 * WAVE - 1) / (4 * WAVE))
void residentKernel(const ResTile * __restrict__ tiles, uint32_t numTiles, const NeuronGroupDev * __restrict__ groups,
                    const uint8_t * __restrict__ tileGroup, unsigned long long *tags, unsigned long long *side,
                    unsigned long long timestep0, unsigned long long epoch0, unsigned long long numRecordingTimesteps, uint32_t numSteps,
                    float dt, uint32_t zeroDelaySplit, uint32_t *errorFlag, unsigned long long *eventCounter, uint32_t replicaStride,
                    unsigned long long seqBase)
{
    extern __shared__ float lds[];                       // inSyn rows and ring slices of this tile
    __shared__ uint2 shSeg[2][RES_PAIR_CAP];             // (first idSyn, length | flags | projection) of each listed pair
    // of an exchange: listed pairs whose row has to be walked before the update; pairs were left over; a wait expired
    struct Taken { uint32_t flagged, left, failed, pad; };
    __shared__ __align__(16) Taken shTaken[4];
    __shared__ uint32_t shDone[4];                       // of the update an exchange feeds: wavefronts done << 16 | spikes
    __shared__ ResProj shProj[RES_MAX_PROJ];
    __shared__ uint32_t shProjPtr[4][RES_MAX_PROJ];      // front slot of each projection's ring in the step an exchange feeds, as a float offset
    __shared__ uint32_t shProjStart[RES_MAX_GROUPS + 1]; // projections of this tile by source group
    __shared__ uint8_t shProjIdx[RES_MAX_PROJ];
    __shared__ uint32_t shOwn[TILE];                    // this tile's spikes of the last step, in no particular order
    constexpr uint32_t THREADS = TILE + WALK * WAVE, WAVES = THREADS / WAVE, MAIN = TILE / WAVE;
    __shared__ uint32_t shWave[WAVES];
    __shared__ uint32_t shListed[4][MAIN];               // pairs each wavefront has listed of an exchange, in its own part of the list
    __shared__ uint32_t shScalar[4];

    // every tile publishes its word into all copies of the word array and reads the copy of its own XCD
    uint32_t xcc = 0;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    const unsigned long long *myTags = tags + (size_t)(xcc & (RES_REPLICAS - 1)) * replicaStride;
    const ResTile &T = tiles[blockIdx.x];
    const NeuronGroupDev &G = groups[T.group];
    const gennmi_neuron_update_group_t &g = G.g;
    const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const uint32_t n = g.numNeurons;
    const uint32_t tileFirst = T.first, tilesInGroup = T.tilesInGroup, tileInGroup = T.tileInGroup;
    const uint32_t i = tileFirst + tid;
    const bool mine = tid < T.count, main = (WALK == 0 || wave < MAIN);
    const uint32_t numPSM = g.numPSM, numCS = g.numCS;

    // (a runner whose error flag is raised launches nothing more: the host looks at the flag before every launch; the flag
    // is host memory, and reading it here would put a trip over the bus in front of every launch)
    // ---- tables into LDS
    const uint32_t numProj = T.numProj;
    if(tid < numProj) { shProj[tid] = T.proj[tid]; }
    if(tid < 4) { shScalar[tid] = 0u; }
    if(tid < 4) { shTaken[tid] = Taken{0u, 0u, 0u, 0u}; shDone[tid] = 0u; }
    __syncthreads();
    // projections grouped by source group (a counting sort of a handful of entries, read from the LDS copy; every thread
    // finds one entry's place by itself — one thread doing all of it is a chain of a hundred dependent LDS reads, 3 us
    // of every launch)
    if(tid <= RES_MAX_GROUPS) {
        uint32_t below = 0;
        for(uint32_t q = 0; q < numProj; q++) { below += (shProj[q].srcGroup < tid) ? 1u : 0u; }
        shProjStart[tid] = below;
    }
    if(tid < numProj) {
        const uint32_t s = shProj[tid].srcGroup;
        uint32_t below = 0, before = 0;
        for(uint32_t q = 0; q < numProj; q++) {
            const uint32_t sq = shProj[q].srcGroup;
            below += (sq < s) ? 1u : 0u;
            before += (q < tid && sq == s) ? 1u : 0u;
        }
        shProjIdx[below + before] = (uint8_t)tid;
        const uint32_t D = shProj[tid].D;
        for(uint32_t e = 1; e <= 2; e++) { shProjPtr[(seqBase + e) & 3][tid] = D ? modStepOnce(epoch0 + e, D) * TILE : 0u; }
    }
    // (lane p < numProj of the last wavefront, which prepares what the exchange after the next needs) front slot of projection p's ring then
    const uint32_t ptrDepth = (wave == WAVES - 1 && lane < numProj) ? max(1u, shProj[lane].D) : 1u;
    uint32_t ptrNext = modStepOnce(epoch0 + 3, ptrDepth);

    // ---- state: neuron variables in registers, inSyn in registers (in LDS where synapses add to it) and ring slices in LDS
    float l0 = 0, l1 = 0;
    if(mine) { l0 = asGlobal(g.var0)[i]; l1 = asGlobal(g.var1)[i]; }
    // state of the PoissonExp sources, in registers like the neuron's own
    float csState[GENNMI_MAX_CS];
    #pragma unroll
    for(uint32_t c = 0; c < GENNMI_MAX_CS; c++) {
        csState[c] = (POISSON && mine && c < numCS && g.cs[c].kind == GENNMI_CS_POISSON_EXP) ? asGlobal(g.cs[c].current)[i] : 0.0f;
    }
    // What the update reads of its group and tile, once: through the references every step would load it again (the
    // compiler cannot tell that nobody writes those structures while the kernel runs), and in vector registers: left to itself the compiler
    // keeps such wave-uniform values in scalar registers, of which there are too few, and fetches them back lane by lane every step.
    auto inVector = [](auto x) { asm volatile("" : "+v"(x)); return x; };
    float psmInit[NPSM], psmDecay[NPSM], csAmp[GENNMI_MAX_CS], par[7], lin[NPSM];
    uint32_t psmExp[NPSM], psmRing[NPSM], psmAt[NPSM], psmEnd[NPSM], csKind[GENNMI_MAX_CS];
    #pragma unroll
    for(uint32_t m = 0; m < NPSM; m++) {
        const bool on = m < numPSM, exponential = on && g.psm[m].kind == GENNMI_PSM_EXPCURR;
        const uint32_t D = on ? g.psm[m].maxDenDelay : 0u;
        psmExp[m] = inVector(exponential ? 1u : 0u); psmRing[m] = inVector(D ? D * TILE : 0u);
        psmInit[m] = inVector(exponential ? g.psm[m].init : 1.0f); psmDecay[m] = inVector(exponential ? g.psm[m].expDecay : 0.0f);
        // this neuron's element of the slot the coming step reads, and one beyond the last slot's; without a ring inSyn itself, in LDS
        psmAt[m] = on ? (D ? T.ldsRing[m] + modStepOnce(epoch0 + 1, D) * TILE : T.ldsIn[m]) + tid : 0u;
        psmEnd[m] = on ? (D ? T.ldsRing[m] + D * TILE : T.ldsIn[m] + 1u) + tid : 0u;
        lin[m] = (on && mine) ? asGlobal(g.psm[m].outPost)[i] : 0.0f;
    }
    #pragma unroll
    for(uint32_t c = 0; c < GENNMI_MAX_CS; c++) { csAmp[c] = (c < numCS) ? g.cs[c].amp : 0.0f; csKind[c] = (c < numCS) ? g.cs[c].kind : 0u; }
    #pragma unroll
    for(uint32_t q = 0; q < 7; q++) { par[q] = inVector(g.params[q]); }
    const bool lif = (g.model == GENNMI_NEURON_LIF);
    GLOBAL_AS uint32_t * const recordSpk = asGlobal(g.recordSpk);
    #pragma unroll
    for(uint32_t m = 0; m < NPSM; m++) {
        if(m >= numPSM) { break; }
        const uint32_t D = g.psm[m].maxDenDelay, ringBase = T.ldsRing[m] + tid;
        // (without a ring synapses add to inSyn itself, and what the register holds of it must add nothing: -0 + x is x, zeros included)
        if(!D) { if(main) { lds[T.ldsIn[m] + tid] = lin[m]; } lin[m] = -0.0f; }
        // (sixteen slots' loads in flight at a time: one at a time, a ring of 43 slots is 43 memory round trips per launch)
        GLOBAL_AS const float *ring = asGlobal(g.psm[m].denDelay) + (mine ? i : 0u);
        for(uint32_t slot0 = 0; slot0 < D; slot0 += 16) {
            float v[16];
            #pragma unroll
            for(uint32_t u = 0; u < 16; u++) { v[u] = (mine && slot0 + u < D) ? ring[(size_t)min(slot0 + u, D - 1) * n] : 0.0f; }
            #pragma unroll
            for(uint32_t u = 0; u < 16; u++) { if(main && slot0 + u < D) { lds[ringBase + (slot0 + u) * TILE] = v[u]; } }
        }
    }

    // ---- this tile's spikes of the step before the first one, from the population's (ascending) queue
    {
        const uint32_t cnt = asGlobal(g.spkCnt)[0];
        uint32_t below = 0, inside = 0;
        for(uint32_t k = tid; k < cnt; k += THREADS) {
            const uint32_t id = asGlobal(g.spk)[k];
            below += (id < tileFirst) ? 1u : 0u;
            inside += (id >= tileFirst && id < tileFirst + T.count) ? 1u : 0u;
        }
        if(below) { atomicAdd(&shScalar[0], below); }
        if(inside) { atomicAdd(&shScalar[1], inside); }
        __syncthreads();
        const uint32_t lo = shScalar[0];
        for(uint32_t k = tid; k < cnt; k += THREADS) {
            const uint32_t id = asGlobal(g.spk)[k];
            if(id >= tileFirst && id < tileFirst + T.count) { shOwn[k - lo] = id; }
        }
    }
    __syncthreads();
    uint32_t ownCount = shScalar[1];

    // (callers synchronise the work-group after filling shOwn)
    // A word slot is rewritten every second sequence number, and a launch continues the numbering of the one before
    // (seqBase), so a slot never holds the number a reader waits for before its writer has stored it: nothing is cleared
    // between launches.  A tile's spikes beyond those its word holds go through the side buffer, one 64-bit entry each that
    // says which exchange it belongs to (the unwrapped sequence number, 54 bits, above the tile-local index): entries and
    // word are stored in any order without a fence, and a reader that finds the word first waits for the entries.
    // (called by one wavefront)
    GLOBAL_AS unsigned long long *tagOut = asGlobal(tags) + (size_t)(lane & (RES_REPLICAS - 1)) * replicaStride + blockIdx.x;
    auto publish = [&](uint32_t step, uint32_t count) {
        const uint32_t seq = (uint32_t)(seqBase + step) & RES_SEQ_MASK, parity = seq & 1u;
        uint32_t locals = 0;
        if(count) {
            if(count > RES_WORD_IDS) {
                for(uint32_t r = lane; r < count; r += WAVE) {
                    __hip_atomic_store(&side[((size_t)parity * numTiles + blockIdx.x) * TILE + r], ((seqBase + step) << RES_ID_BITS) | (shOwn[r] - tileFirst),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            for(uint32_t e = 0; e < min(count, RES_WORD_IDS); e++) { locals |= (shOwn[e] - tileFirst) << (RES_ID_BITS * e); }
        }
        const unsigned long long word = ((unsigned long long)((seq << RES_COUNT_BITS) | count) << 32) | locals;
        if(lane < RES_REPLICAS) { __hip_atomic_store(tagOut + (parity ? numTiles : 0u), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    };

    // The source tile this thread watches and the spikes it takes of it: all of them, or, where there are fewer tiles than half the threads,
    // those that fall to it among the threads that watch the same one.
    uint32_t perTile = 1, perShift = 0, watchTile = tid, watchSub = 0;
    // (entries of eight quads are read by eight lanes each: with few enough tiles the eight watch the same one, `grouped`)
    bool grouped = QUADS == RES_MAX_QUADS && numTiles <= TILE / RES_MAX_QUADS;
    for(uint32_t q = 0; grouped && q < numProj; q++) { grouped = shProj[q].D == 0; }
    if(grouped) {
        const uint32_t shift = 32u - (uint32_t)__clz(max(numTiles, 2u) - 1u), group = tid / RES_MAX_QUADS;
        perTile = (TILE / RES_MAX_QUADS) >> shift;
        watchTile = group & ((1u << shift) - 1u); watchSub = group >> shift;
    }
    else if((TILE & (TILE - 1)) == 0 && numTiles <= TILE / 2) {
        const uint32_t shift = 32u - (uint32_t)__clz(max(numTiles, 2u) - 1u);       // (tiles rounded up to a power of two)
        perTile = TILE >> shift; perShift = 31u - (uint32_t)__clz(perTile);
        watchTile = tid & ((1u << shift) - 1u); watchSub = tid >> shift;
    }
    const bool watching = main && watchTile < numTiles;
    // The list is shared out between the wavefronts that watch: a pair's place depends on the spikes alone and not on when their words
    // arrive, so a wavefront that walks adds the synapses of an exchange in the same order every time.  Between wavefronts there is no order, nor for
    // the due synapses, which the thread that sees a word adds: sums that round differ from run to run.  (Where places followed the words' arrival,
    // two runs of the full microcircuit parted at every neuron that comes within a rounding of its threshold.  As it is, 24 runs of 10,000 steps, four
    // of each of six seeds, had the same rasters and membranes that differ by 1.5e-5 mV.)
    const uint32_t watchWaves = (perTile == 1) ? (numTiles + WAVE - 1) / WAVE : MAIN, listCap = RES_PAIR_CAP / watchWaves;
    const uint32_t rowQuads = QUADS * tilesInGroup;     // entries of consecutive rows, in quads
    const uint32_t watchFirst = watching ? tiles[watchTile].first : 0u;
    uint32_t watchProj0 = 0, watchNumProj = 0, watchLds = 0, watchFlags = 0;             // (flags: the first projection's number << 26)
    GLOBAL_AS const u32x4 *watchSeg = nullptr;           // entry of the tile's first neuron under its group's first projection into this tile
    if(watching) {
        const uint32_t s = tileGroup[watchTile];
        watchProj0 = shProjStart[s];
        watchNumProj = shProjStart[s + 1] - watchProj0;
        if(watchNumProj) {
            const uint32_t p = shProjIdx[watchProj0];
            watchSeg = asGlobal(shProj[p].seg) + QUADS * ((size_t)watchFirst * tilesInGroup + tileInGroup);
            watchFlags = p << RES_SEG_PROJ_SHIFT;
            watchLds = shProj[p].lds;
        }
    }

    // entries of a side list that are asked for at a time
    constexpr uint32_t FLIGHT = 3;
    // Entries e0, e0 + perTile, ... (FLIGHT of them, below c) of the watched tile's side list of the exchange `full`: waits, bounded, until each says so
    auto sideIds = [&](uint32_t e0, uint32_t c, unsigned long long full, uint32_t parity, uint32_t (&local)[FLIGHT]) -> bool {
        const unsigned long long *base = side + ((size_t)parity * numTiles + watchTile) * TILE + e0;
        const unsigned long long want = full & (~0ull >> RES_ID_BITS);
        uint32_t need = 0, spins = 0;
        #pragma unroll
        for(uint32_t u = 0; u < FLIGHT; u++) { if(e0 + u * perTile < c) { need |= 1u << u; } }
        unsigned long long v[FLIGHT];
        while(true) {
            #pragma unroll
            for(uint32_t u = 0; u < FLIGHT; u++) { v[u] = 0; if(need & (1u << u)) { v[u] = __hip_atomic_load(base + u * perTile, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); } }
            #pragma unroll
            for(uint32_t u = 0; u < FLIGHT; u++) {
                if((need & (1u << u)) && (v[u] >> RES_ID_BITS) == want) { local[u] = (uint32_t)v[u] & RES_ID_MASK; need &= ~(1u << u); }
            }
            if(!need) { return true; }
            if(++spins > c_spinLimit) { return false; }
            __builtin_amdgcn_s_sleep(1);
        }
    };

    unsigned long long events = 0;

    constexpr uint32_t PASS_ALL = 0, PASS_LATER = 1, PASS_DUE = 2, PASS_NONE = 3;      // which synapses a pass adds: see process()

    struct Entry { u32x4 quad[QUADS]; };
    auto readEntry = [&](GLOBAL_AS const u32x4 *entry) -> Entry {
        Entry e;
        #pragma unroll
        for(uint32_t q = 0; q < QUADS; q++) { e.quad[q] = entry[q]; }
        return e;
    };
    // What a segment entry says: lists the pair and — unless `skipInline` — adds the synapses inside to the front slot
    auto takeEntry = [&](const Entry &e, uint32_t flags, uint32_t frontBase, uint32_t slot, uint32_t pos, bool skipInline, bool count) {
        const uint32_t head = e.quad[0].y;
        shSeg[slot & 1][pos] = make_uint2(e.quad[0].x, head | flags);
        if(head & RES_SEG_OVERFLOW) { atomicAdd(&shTaken[slot].flagged, 1u); }
        if(count) { events += head & 0xFFFFu; }
        const uint32_t inside = skipInline ? 0u : (head >> 16) & 0xFFu;
        #pragma unroll
        for(uint32_t q = 0; q < QUADS; q++) {
            if(!__any((q ? 3 * q - 2 : 0u) < inside)) { break; }
            const u32x4 x = e.quad[q];
            const float w[3] = {__uint_as_float(q ? x.x : x.z), __uint_as_float(x.y), __uint_as_float(x.z)};
            #pragma unroll
            for(uint32_t f = 0; f < (q ? 3u : 1u); f++) {
                if((q ? 3 * q - 2 : 0u) + f < inside) { unsafeAtomicAdd(&lds[frontBase + ((x.w >> (RES_ID_BITS * f)) & RES_ID_MASK)], w[f]); }
            }
        }
    };
    // An entry of eight quads, by eight consecutive lanes with the same arguments: a quad each, and each adds its synapses.  A row part that is longer
    // than an entry is walked on the spot (without a ring all of it is due).  (Nothing is listed: there is nothing left for later.)
    auto takeTogether = [&](uint32_t id, uint32_t p, bool skipInline, bool count) {
        const ResProj &P = shProj[p];
        const uint32_t u = lane & (RES_MAX_QUADS - 1), base = P.lds;
        const u32x4 x = (asGlobal(P.seg) + RES_MAX_QUADS * ((size_t)id * tilesInGroup + tileInGroup))[u];
        const uint32_t n = skipInline ? 0u : x.w >> RES_COUNT_SHIFT;
        const float w[3] = {__uint_as_float(u ? x.x : x.z), __uint_as_float(x.y), __uint_as_float(x.z)};
        #pragma unroll
        for(uint32_t f = 0; f < 3; f++) {
            if(f < n) { unsafeAtomicAdd(&lds[base + ((x.w >> (RES_ID_BITS * f)) & RES_ID_MASK)], w[f]); }
        }
        if(count && u == 0) { events += x.y & 0xFFFFu; }
        const uint32_t head = __shfl(x.y, 0, RES_MAX_QUADS), start = __shfl(x.x, 0, RES_MAX_QUADS);
        if((head & RES_SEG_OVERFLOW) && !skipInline) {
            GLOBAL_AS const u32x2 *packed = asGlobal(P.packed) + start;
            for(uint32_t r = u; r < (head & 0xFFFFu); r += RES_MAX_QUADS) {
                const u32x2 rec = packed[r];
                unsafeAtomicAdd(&lds[base + rec.x / 4u], __uint_as_float(rec.y));
            }
        }
    };

    // Waits for every tile's word of exchange `step` (main threads; shTaken says when the bounded wait expired somewhere) and takes the
    // (spike, projection) pairs that concern this tile: lists them and — `convention` PASS_ALL or PASS_DUE — adds the due synapses
    // their entries hold.  Pairs that find no place in the list are left to leftOver() (`left`: this thread's are).
    unsigned long long word = 0;
    bool left = false;
    auto spikesOf = [&]() -> uint32_t { return (uint32_t)(word >> 32) & RES_COUNT_MASK; };
    auto idOf = [&](uint32_t e) -> uint32_t { return ((uint32_t)word >> (RES_ID_BITS * e)) & RES_ID_MASK; };        // (e < RES_WORD_IDS)
    // Cycles from a tile's own word to its first look for the others'.  A look that comes too early costs its whole trip to memory again, and
    // the looks of all the waiting tiles slow the words down: the more tiles, the longer the words take.  us a step without the wait / with 1,000 /
    // 1,500 / 2,000 cycles / as below: 20,000 x 100 (79 tiles) 2.76 / 2.37 / 2.42 / 2.62 / 2.35, 40,000 x 80 (157) 3.79 / 3.29 / 3.24 / 3.41 / 3.25,
    // 100,000 x 80 (196) 4.83 / 4.30 / 4.04 / 4.05 / 4.05, the full microcircuit (243) 4.66 / 4.23 / - / - / 4.09.  A handful of tiles are too quick for it
    // (1,000 x 80 2.10 / 2.17).  Drawing of Poisson sources takes longer than the wait.
    const uint32_t firstLook = (numTiles <= 8) ? 0u : min(800u + 4u * numTiles, 1700u);
    uint32_t published = (uint32_t)__builtin_readcyclecounter();
    auto poll = [&](uint32_t step, uint32_t convention) {
        const uint32_t seq = (uint32_t)(seqBase + step) & RES_SEQ_MASK;
        const uint32_t parity = seq & 1u, slot = seq & 3u;
        const bool skipInline = (convention == PASS_LATER), count = (convention != PASS_DUE);
        bool ok = true;
        left = false;
        word = 0;
        if(watching) {
            const unsigned long long *mine_ = myTags + (parity ? numTiles : 0u) + watchTile;
            uint32_t spins = 0;
            while((uint32_t)__builtin_readcyclecounter() - published < firstLook) { __builtin_amdgcn_s_sleep(1); }
            while(true) {
                word = __hip_atomic_load(mine_, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if((uint32_t)(word >> (32 + RES_COUNT_BITS)) == seq) { break; }
                ++spins;
                if(spins > c_spinLimit || ((spins & 255u) == 0 && __hip_atomic_load(errorFlag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) { ok = false; word = 0; break; }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        const uint32_t c = spikesOf();
        uint32_t listed = 0;
        if(convention != PASS_NONE && __any(c != 0u)) {
            if(grouped) {
                for(uint32_t e = watchSub; e < c && ok; e += perTile) {
                    uint32_t local[FLIGHT] = {};
                    if(c <= RES_WORD_IDS) { local[0] = idOf(e); }
                    else if(!sideIds(e, min(c, e + 1), seqBase + step, parity, local)) { ok = false; }
                    for(uint32_t j = 0; ok && j < watchNumProj; j++) { takeTogether(watchFirst + local[0], shProjIdx[watchProj0 + j], skipInline, count); }
                }
            }
            else {
                // this thread's pairs
                const uint32_t mineCount = (c > watchSub && watchNumProj != 0) ? ((c - watchSub + perTile - 1) >> perShift) : 0u, total = mineCount * watchNumProj;
                const uint32_t listBase = wave * listCap;
                const unsigned long long busy = __ballot(total != 0u);
                listed = __popcll(busy);
                if(__any(total > 1u || (total != 0u && c > RES_WORD_IDS))) {         // (beyond RES_WORD_IDS the ids are in the side list)
                    // Some thread of the wavefront has many pairs: the wavefront lists its pairs first and every
                    // lane then takes as many of them as every other, so that their entries are one trip to memory and not one after another.
                    const uint32_t inclusive = waveInclusiveScanU32(total, lane);
                    listed = (uint32_t)__builtin_amdgcn_readlane((int)inclusive, WAVE - 1);
                    const bool fits = (listed <= listCap);
                    uint32_t pos = listBase + inclusive - total;
                    left = !fits && total != 0;
                    for(uint32_t e0 = watchSub; total != 0 && e0 < c && ok; e0 += FLIGHT * perTile) {
                        uint32_t local[FLIGHT];
                        #pragma unroll
                        for(uint32_t u = 0; u < FLIGHT; u++) { local[u] = (e0 + u * perTile < RES_WORD_IDS) ? idOf(e0 + u * perTile) : 0u; }
                        // (also when the pairs do not fit and leftOver() will read the list again: once seen here, an entry is there
                        // for every later read of this thread)
                        if(c > RES_WORD_IDS && !sideIds(e0, c, seqBase + step, parity, local)) { ok = false; }
                        #pragma unroll
                        for(uint32_t u = 0; u < FLIGHT; u++) {
                            if(!fits || e0 + u * perTile >= c) { break; }
                            for(uint32_t j = 0; j < watchNumProj; j++) { shSeg[slot & 1][pos++] = make_uint2(watchFirst + local[u], shProjIdx[watchProj0 + j]); }
                        }
                    }
                    if(!fits) {
                        listed = 0;
                        if(lane == 0) { shTaken[slot].left = 1u; }
                    }
                    else if(!__any(!ok)) {
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                        for(uint32_t x = listBase + lane; x < listBase + listed; x += WAVE) {
                            const uint2 pr = shSeg[slot & 1][x];
                            const ResProj &P = shProj[pr.y];
                            takeEntry(readEntry(asGlobal(P.seg) + QUADS * ((size_t)pr.x * tilesInGroup + tileInGroup)), pr.y << RES_SEG_PROJ_SHIFT, P.lds + shProjPtr[slot][pr.y], slot, x, skipInline, count);
                        }
                    }
                }
                else {
                    // (what nearly every quiet step has: at most one pair a thread.  Handling up to three here, unrolled or in a loop, made the
                    // step slower whether it had them or not)
                    if(total) {
                        takeEntry(readEntry(watchSeg + (size_t)idOf(watchSub) * rowQuads), watchFlags, watchLds + shProjPtr[slot][watchFlags >> RES_SEG_PROJ_SHIFT],
                                  slot, listBase + __popcll(busy & ((1ull << lane) - 1ull)), skipInline, count);
                    }
                }
            }
        }
        if(lane == 0) { shListed[slot][wave] = listed; }
        if(!ok) { shTaken[slot].failed = 1u; }
    };

    // Walks the row segments of the listed pairs: a group of lanes per pair, a lane taking every n-th synapse of its
    // pair's segment, four of them per trip to memory.  Sixteen lanes per pair when the pairs are few (a quiet step: one
    // trip covers 64 synapses of each of a wavefront's four pairs), four when they are many (a synchronous burst).
    // (Segments are short — a row's share of a tile's targets — so lanes idle in the longest segment's last trip
    // cost less than finding, for every lane, its place in a list of all the segments' synapses would.)
    // A synapse is "due" when it lands in the slot read this step (delay a multiple of the ring depth, or no ring).
    // PASS_ALL adds every synapse, PASS_LATER those not due, PASS_DUE the due ones; `flaggedOnly` restricts the walk to
    // segments whose due synapses are not all inline in their entry.
    // (wavefront `first` of the `count` that call; pair q is in segs[place(q)], which all lanes ask for together)
    auto process = [&](const uint2 *segs, auto place, const uint32_t *fronts, uint32_t numPairs, uint32_t pass, bool flaggedOnly, uint32_t first, uint32_t count) {
        constexpr uint32_t TRIP = 4, DUE_END = 4 * TILE;
        const uint32_t from = (pass == PASS_LATER) ? DUE_END : 0u, span = (pass == PASS_DUE) ? DUE_END : 0xFFFFFFFFu - from;      // offsets that are added
        const uint32_t shift = (numPairs <= 4 * count) ? 4u : (numPairs <= 8 * count) ? 3u : 2u;
        const uint32_t lanesPerPair = 1u << shift, pairsPerGroup = WAVE >> shift;
        for(uint32_t q0 = first * pairsPerGroup; q0 < numPairs; q0 += count * pairsPerGroup) {
            const uint32_t q = q0 + (lane >> shift), at = place(min(q, numPairs - 1u));
            uint32_t len = 0, start = 0, proj = 0;
            if(q < numPairs) {
                const uint2 sg = segs[at];
                proj = sg.y >> RES_SEG_PROJ_SHIFT;
                const bool flagged = (sg.y & RES_SEG_OVERFLOW) != 0;
                const bool skip = (flaggedOnly && !flagged) || (pass == PASS_LATER && (sg.y & RES_SEG_NO_DELAY));
                len = skip ? 0u : (sg.y & 0xFFFFu);
                start = len ? sg.x : 0u;                          // (an empty part may start where the array ends)
            }
            const ResProj &P = shProj[proj];
            const uint32_t front = 4u * fronts[proj], ringBytes = 4u * TILE * P.D, ldsBase = 4u * P.lds;
            GLOBAL_AS const u32x2 *packed = asGlobal(P.packed) + start;
            const uint32_t last = len ? len - 1u : 0u;
            for(uint32_t i0 = lane & (lanesPerPair - 1); __any(i0 < len); i0 += TRIP * lanesPerPair) {
                // (a lane beyond the part's end reads its last record again: no branch between the loads)
                u32x2 rec[TRIP];
                #pragma unroll
                for(uint32_t u = 0; u < TRIP; u++) { rec[u] = packed[min(i0 + u * lanesPerPair, last)]; }
                #pragma unroll
                for(uint32_t u = 0; u < TRIP; u++) {
                    uint32_t at = front + rec[u].x;                          // (a multiple of four below twice the ring's bytes)
                    at = min(at, at - ringBytes);                             // (at < ringBytes: the difference wraps round)
                    if(i0 + u * lanesPerPair < len && rec[u].x - from < span) {
                        unsafeAtomicAdd(reinterpret_cast<float*>(reinterpret_cast<char*>(lds) + (ldsBase + at)), __uint_as_float(rec[u].y));
                    }
                }
            }
        }
    };

    // The pairs that found no place in the list: listed and walked RES_PAIR_CAP at a time, in full, before the
    // update (in the other parity's list: its pairs were walked before this exchange's words were looked for, and the next
    // exchange's threads come here first).
    auto leftOver = [&](uint32_t step, uint32_t pass, bool count) {
        const uint32_t slot = (uint32_t)(seqBase + step) & 3u, parity = slot & 1u, other = parity ^ 1u;
        const uint32_t c = spikesOf(), want = left ? ((c - watchSub + perTile - 1) >> perShift) * watchNumProj : 0u;
        const uint32_t inclusive = waveInclusiveScanU32(want, lane);
        if(lane == WAVE - 1) { shWave[wave] = inclusive; }
        __syncthreads();
        uint32_t base = inclusive - want, total = 0;
        #pragma unroll
        for(uint32_t w = 0; w < WAVES; w++) { if(w < wave) { base += shWave[w]; } total += shWave[w]; }
        for(uint32_t chunk0 = 0; chunk0 < total; chunk0 += RES_PAIR_CAP) {
            uint32_t pos = base;
            if(left && pos + want > chunk0 && pos < chunk0 + RES_PAIR_CAP) {
                for(uint32_t e = watchSub; e < c; e += perTile) {
                    const uint32_t id = watchFirst + ((c <= RES_WORD_IDS) ? idOf(e)
                                                                          : (uint32_t)__hip_atomic_load(&side[((size_t)parity * numTiles + watchTile) * TILE + e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & RES_ID_MASK);
                    for(uint32_t j = 0; j < watchNumProj; j++, pos++) {
                        if(pos >= chunk0 && pos < chunk0 + RES_PAIR_CAP) { shSeg[other][pos - chunk0] = make_uint2(id, shProjIdx[watchProj0 + j]); }
                    }
                }
            }
            __syncthreads();
            const uint32_t numPairs = min(RES_PAIR_CAP, total - chunk0);
            for(uint32_t q = tid; q < numPairs; q += THREADS) {
                const uint2 pr = shSeg[other][q];
                const ResProj &P = shProj[pr.y];
                const u32x4 lo4 = (asGlobal(P.seg) + QUADS * ((size_t)pr.x * tilesInGroup + tileInGroup))[0];
                shSeg[other][q] = make_uint2(lo4.x, (lo4.y & ~(0x3Fu << RES_SEG_PROJ_SHIFT)) | (pr.y << RES_SEG_PROJ_SHIFT));
                if(count) { events += lo4.y & 0xFFFFu; }
            }
            __syncthreads();
            process(shSeg[other], [](uint32_t q) { return q; }, shProjPtr[slot], numPairs, pass, false, wave, WAVES);
            __syncthreads();
        }
    };

    // After poll(), by all threads: the barrier, and whatever the listed entries could not deliver at once.  `convention` is PASS_ALL
    // normally, PASS_LATER when a previous launch has already delivered the due synapses of these spikes, PASS_DUE when only those
    // are wanted.  False: some wait expired.
    auto walkListed = [&](uint32_t slot, uint32_t pass, bool flaggedOnly, uint32_t first, uint32_t count) {
        // (pair q of the wavefronts' parts one after the other)
        uint32_t upTo = (lane < watchWaves) ? shListed[slot][lane] : 0u;
        #pragma unroll
        for(uint32_t d = 1; d < MAIN; d <<= 1) {
            const uint32_t below = __shfl_up(upTo, d);
            upTo += (lane >= d) ? below : 0u;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)upTo, MAIN - 1);
        auto place = [&](uint32_t q) {
            uint32_t part = 0, before = 0;
            #pragma unroll
            for(uint32_t half = (MAIN > 8) ? 8 : (MAIN > 4) ? 4 : 2; half != 0; half /= 2) {
                const uint32_t x = __shfl(upTo, part + half - 1);
                before = (x <= q) ? x : before;
                part = (x <= q) ? part + half : part;
            }
            return part * listCap + q - before;
        };
        if(total) { process(shSeg[slot & 1], place, shProjPtr[slot], total, pass, flaggedOnly, first, count); }
    };
    auto deliverDue = [&](uint32_t step, uint32_t convention) -> bool {
        const uint32_t slot = (uint32_t)(seqBase + step) & 3u;
        ldsBarrier();
        Taken taken = shTaken[slot];
        taken.flagged = __builtin_amdgcn_readfirstlane(taken.flagged);
        taken.left = __builtin_amdgcn_readfirstlane(taken.left); taken.failed = __builtin_amdgcn_readfirstlane(taken.failed);
        if(taken.flagged | taken.left | taken.failed) {
            if(taken.failed) {
                if(tid == 0) { raiseErrorFlag(errorFlag); }
                return false;
            }
            if(convention != PASS_LATER && taken.flagged) { walkListed(slot, PASS_DUE, true, wave, WAVES); ldsBarrier(); }
            if(taken.left) { leftOver(step, convention, convention != PASS_DUE); }
        }
        return true;
    };

    bool anyRing = false;
    for(uint32_t q = 0; q < numProj; q++) { anyRing = anyRing || shProj[q].D != 0; }
    // where the coming step's recording word of this half wavefront goes, and the steps until the buffer wraps
    const unsigned long long recT = numRecordingTimesteps ? (((timestep0 | numRecordingTimesteps) >> 32) ? timestep0 % numRecordingTimesteps
                                                                                                          : (uint32_t)timestep0 % (uint32_t)numRecordingTimesteps) : 0ull;
    const uint32_t recordWords = numRecordingTimesteps ? (n + 31) / 32 : 0u;
    const bool recordHere = recordSpk != nullptr && (lane & 31) == 0 && mine;
    GLOBAL_AS uint32_t *recordAt = recordSpk + (size_t)recT * recordWords + (i >> 5);
    uint32_t recordLeft = (uint32_t)min(numRecordingTimesteps - recT, 0xFFFFFFFFull);       // (a launch has fewer steps than this can count)
    // ---- exchange the spikes that precede the first step, then step
    if(wave == 0) { publish(1u, ownCount); }
    bool ok = true;
    uint32_t k = 0;
    for(; k < numSteps; k++) {
        const unsigned long long epoch = epoch0 + k;
        const uint32_t slot = (uint32_t)(seqBase + k + 1) & 3u, afterNext = (slot + 2) & 3u;
        const uint32_t convention = (zeroDelaySplit && k == 0) ? PASS_LATER : PASS_ALL;
        float inject[GENNMI_MAX_CS];
        if(main) {
            // (what the sources inject does not depend on the exchange: drawn while the words travel)
            #pragma unroll
            for(uint32_t c = 0; c < GENNMI_MAX_CS; c++) {
                inject[c] = 0.0f;
                if(POISSON && c < numCS) { inject[c] = (csKind[c] == GENNMI_CS_DC) ? csAmp[c] : (mine ? poissonExpStep(g.cs[c], csState[c], i, epoch) : 0.0f); }
            }
            poll(k + 1, convention);
        }
        if(!deliverDue(k + 1, convention)) { ok = false; break; }
        if(wave == WAVES - 1) {
            if(lane < numProj) { shProjPtr[afterNext][lane] = ptrNext * TILE; }
            if(lane == 0) { shTaken[afterNext] = Taken{0u, 0u, 0u, 0u}; shDone[afterNext] = 0u; }
            ptrNext = (ptrNext + 1 >= ptrDepth) ? 0u : ptrNext + 1;
        }
        if(main) {
        // neuron update: same operations in the same order as neuronBody, as selections instead of branches
        bool spiked = false;
        float Isyn = 0;
        #pragma unroll
        for(uint32_t m = 0; m < NPSM; m++) {
            if(m >= numPSM) { break; }
            const bool ring = (psmRing[m] != 0u);
            const float linSyn = lin[m] + lds[psmAt[m]];
            const float decayed = psmExp[m] ? linSyn * psmDecay[m] : 0.0f;
            Isyn += psmInit[m] * linSyn;
            lds[psmAt[m]] = ring ? 0.0f : decayed;
            lin[m] = ring ? decayed : -0.0f;
        }
        #pragma unroll
        for(uint32_t c = 0; c < GENNMI_MAX_CS; c++) {
            if(c >= numCS) { break; }
            Isyn += POISSON ? inject[c] : csAmp[c];
        }
        if(lif) {
            const bool active = (l1 <= 0.0f);
            const float alpha = ((Isyn + par[0]) * par[1]) + par[2];
            l0 = active ? alpha - (par[3] * (alpha - l0)) : l0;
            l1 = active ? l1 : l1 - dt;
            spiked = (mine && l1 <= 0.0f && l0 >= par[4]);
            l0 = spiked ? par[5] : l0; l1 = spiked ? par[6] : l1;
        }
        else {
            const bool reset = (l0 >= 30.0f);
            l0 = reset ? par[2] : l0; l1 = reset ? l1 + par[3] : l1;
            l0 += 0.5f * (0.04f * l0 * l0 + 5.0f * l0 + 140.0f - l1 + Isyn) * dt;
            l0 += 0.5f * (0.04f * l0 * l0 + 5.0f * l0 + 140.0f - l1 + Isyn) * dt;
            l1 += par[0] * (par[1] * l0 - l1) * dt;
            l0 = (l0 > 30.0f) ? 30.0f : l0;
            spiked = (mine && l0 >= 29.99f);
        }
        // (a wavefront without spikes, which nearly all are, only says that it is done)
        const unsigned long long ballot = __ballot(spiked);
        if(ballot) {
            uint32_t base = 0;
            if(lane == 0) { base = atomicAdd(&shDone[slot], (uint32_t)__popcll(ballot)); }
            base = __builtin_amdgcn_readfirstlane(base) & 0xFFFFu;
            if(spiked) { shOwn[base + __popcll(ballot & ((1ull << lane) - 1ull))] = i; }
        }
        if(WALK) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            uint32_t done = 0;
            if(lane == 0) { done = atomicAdd(&shDone[slot], 1u << 16); }
            done = __builtin_amdgcn_readfirstlane(done);
            if((done >> 16) == MAIN - 1) {
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                publish(k + 2, done & 0xFFFFu);
            }
        }
        else {
            ldsBarrier();
            if(wave == 0) { publish(k + 2, shDone[slot]); }
        }
        published = (uint32_t)__builtin_readcyclecounter();
        // while the words of this step travel: the step's recording words, and (next) the synapses of the previous step's spikes
        // that are not due yet
        if(recordHere) { *recordAt = (lane & 32) ? (uint32_t)(ballot >> 32) : (uint32_t)ballot; }
        recordAt += recordWords;
        if(--recordLeft == 0u) { recordAt = recordSpk + (i >> 5); recordLeft = (uint32_t)min(numRecordingTimesteps, 0xFFFFFFFFull); }
        #pragma unroll
        for(uint32_t m = 0; m < NPSM; m++) {
            if(m >= numPSM) { break; }
            const uint32_t next = psmAt[m] + TILE;
            psmAt[m] = (next >= psmEnd[m]) ? psmAt[m] + (psmRing[m] ? TILE - psmRing[m] : 0u) : next;
        }
        }
        if((WALK == 0 || !main) && anyRing) {       // (without a ring nothing is: the next word is looked for at once)
            walkListed(slot, PASS_LATER, false, WALK ? wave - MAIN : wave, WALK ? WALK : MAIN);
        }
    }

    // ---- after the last step: everybody's last spikes give the position of this tile's spikes in the population's
    // queue; a runner that delivers front-slot synapses one step early (single-launch plan) wants them in the ring now
    const unsigned long long epochEnd = epoch0 + numSteps;       // completed steps
    if(!ok) { return; }
    const uint32_t lastConvention = zeroDelaySplit ? PASS_DUE : PASS_NONE;
    if(main) { poll(numSteps + 1, lastConvention); }
    if(!deliverDue(numSteps + 1, lastConvention)) { return; }
    __syncthreads();
    ownCount = shDone[(uint32_t)(seqBase + numSteps) & 3u] & 0xFFFFu;       // (the last update's)

    if(mine) {
        asGlobal(g.var0)[i] = l0; asGlobal(g.var1)[i] = l1;
        #pragma unroll
        for(uint32_t c = 0; c < GENNMI_MAX_CS; c++) {
            if(POISSON && c < numCS && g.cs[c].kind == GENNMI_CS_POISSON_EXP) { asGlobal(g.cs[c].current)[i] = csState[c]; }
        }
    }
    #pragma unroll
    for(uint32_t m = 0; m < NPSM; m++) {
        if(m >= numPSM) { break; }
        const uint32_t D = g.psm[m].maxDenDelay;
        if(mine) { asGlobal(g.psm[m].outPost)[i] = D ? lin[m] : lds[T.ldsIn[m] + tid]; }
        for(uint32_t slot = 0; slot < D; slot++) {
            if(mine) { asGlobal(g.psm[m].denDelay)[(size_t)slot * n + i] = lds[T.ldsRing[m] + slot * TILE + tid]; }
        }
        if(tileInGroup == 0 && tid == 0 && D && g.psm[m].denDelayPtr) { *g.psm[m].denDelayPtr = modStepOnce(epochEnd, D); }
    }
    uint32_t offset = (watching && watchSub == 0 && !(grouped && (lane & (RES_MAX_QUADS - 1)) != 0) && watchTile >= T.firstTileOfGroup && watchTile < T.firstTileOfGroup + tileInGroup) ? spikesOf() : 0u;
    if(tid == 0) { shScalar[2] = 0; }
    __syncthreads();
    if(offset) { atomicAdd(&shScalar[2], offset); }
    __syncthreads();
    offset = shScalar[2];
    const bool lastTile = (tileInGroup == tilesInGroup - 1);
    const uint32_t shadowParity = (uint32_t)((epochEnd - 1) & 1);
    for(uint32_t r = tid; r < ownCount; r += THREADS) {
        const uint32_t id = shOwn[r];
        uint32_t place = offset;                         // (queues ascend)
        for(uint32_t q = 0; q < ownCount; q++) { place += (shOwn[q] < id) ? 1u : 0u; }
        g.spk[place] = id;
        for(uint32_t q = 0; q < g.numExtraSpk; q++) { g.extraSpk[q][place] = id; }
        if(G.shadowSpk) { G.shadowSpk[(size_t)shadowParity * n + place] = id; }
    }
    if(lastTile && tid == 0) {
        g.spkCnt[0] = offset + ownCount;
        for(uint32_t q = 0; q < g.numExtraSpk; q++) { g.extraSpkCnt[q][0] = offset + ownCount; }
        if(G.shadowSpk) { G.shadowCnt[shadowParity] = offset + ownCount; }
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) { events += __shfl_down(events, off, WAVE); }
    if(lane == 0 && events) { addEvents(eventCounter, events); }
}


#endif
