// How aheadConvKernel's work-groups share out a layer's output rows and what each keeps in LDS (host code and the kernel; plain C++).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace
{
constexpr uint32_t AHEAD_WORD = 32;             // steps per word (rows of a product)
// A work-group of the convolution takes no more output rows than leave two of them to a compute unit; a single row may take a little more.
constexpr size_t AHEAD_ROWS_LDS = 64 * 1024, AHEAD_MAX_LDS = 82 * 1024;
// Work-groups of a compute unit: four by their registers, and by 160 KiB of LDS, given out in parts of 1,280 bytes.
constexpr uint32_t AHEAD_CONV_GROUPS = 4, AHEAD_CONV_WAVES = 4;
constexpr size_t AHEAD_CU_LDS = 160 * 1024, AHEAD_LDS_PART = 1280, AHEAD_CONV_STATIC_LDS = 288;

// Most inputs with a spike in one step that a list of a pixel's step holds.
constexpr uint32_t AHEAD_CONV_MOST = 16;
// bytes of a wavefront's lists: of a pixel's active inputs, all of them and what fills the last pair; or of the active inputs of its two pixels in each of
// 32 steps, `depth` of 16 bits each
constexpr uint32_t aheadConvListBytes(uint32_t inputs, uint32_t depth)
{
    const uint32_t pixel = 8u * (inputs + 1u), steps = 2u * AHEAD_WORD * depth * 2u;
    return (pixel > steps) ? pixel : steps;
}
// (a row of zeros behind the kernel fills the lists of steps up; `place` has 16 bits an input)
constexpr size_t aheadConvBytes(uint32_t inputs, uint32_t patchWords, uint32_t depth)
{
    return ((size_t)patchWords + (size_t)(inputs + (depth ? 1u : 0u)) * 32 + (inputs + 1) / 2) * sizeof(uint32_t) + (size_t)AHEAD_CONV_WAVES * aheadConvListBytes(inputs, depth);
}
constexpr uint32_t aheadConvResident(size_t bytes)
{
    const size_t parts = (bytes + AHEAD_CONV_STATIC_LDS + AHEAD_LDS_PART - 1) / AHEAD_LDS_PART, fit = AHEAD_CU_LDS / (parts * AHEAD_LDS_PART);
    return (fit < AHEAD_CONV_GROUPS) ? (uint32_t)fit : AHEAD_CONV_GROUPS;
}

struct AheadConvLayout
{
    uint32_t rowsPerBlock, rowPitch;        // output rows of a work-group; words of a patch row
    uint32_t listDepth;                     // inputs that a list of a step holds (0: sums are products throughout)
    size_t bytes;                           // of LDS
    bool fits;
};
// As many output rows per work-group as leave four work-groups to a compute unit, within LDS.  A step's list is as deep as the sums made one by one have use for
// (a quarter of the inputs, AHEAD_CONV_MOST at most), but costs no compute unit a work-group that the launch has for it: with lists of 16 whatever they
// displaced, 50 steps of batch 16 at 0.5 / 2.5 / 10 / 30 %, 64x40x8 -> 32 5x5, 142 / 238 / 350 / 400 us without lists became 183 / 229 / 404 / 457 (three work-groups a
// unit instead of four), 64x72x16 -> 32 3x3 206 / 330 / 503 / 622 became 257 / 326 / 570 / 693.
constexpr AheadConvLayout aheadConvLayout(int32_t kh, int32_t kw, int32_t ic, int32_t oh, int32_t ow, int32_t oc, uint32_t batch, uint32_t numCU)
{
    // (an input takes at least 166 bytes: weights, place, list and patch.  So a weight's place in the kernel, 128 bytes each, always fits a list's 16 bits)
    static_assert((AHEAD_MAX_LDS / 166 + 1) * 128 < 65536, "places of weights in lists have 16 bits");
    AheadConvLayout L{};
    const uint32_t inputs = (uint32_t)(kh * kw * ic);
    L.rowPitch = (uint32_t)(ow - 1 + kw) * (uint32_t)ic;
    const uint64_t columns = (uint64_t)batch * (((uint32_t)oc + 31) / 32), rows = (uint64_t)oh * columns / (4 * numCU);
    L.rowsPerBlock = (rows < 1) ? 1u : (rows < (uint64_t)oh) ? (uint32_t)rows : (uint32_t)oh;
    for(;; L.rowsPerBlock--) {
        L.bytes = aheadConvBytes(inputs, (L.rowsPerBlock + kh - 1) * L.rowPitch, 0);
        if(L.bytes <= AHEAD_ROWS_LDS || L.rowsPerBlock == 1) { break; }
    }
    L.fits = (L.bytes <= AHEAD_MAX_LDS);
    const uint64_t groups = ((uint32_t)oh + L.rowsPerBlock - 1) / L.rowsPerBlock * columns, perUnit = (groups + numCU - 1) / numCU;
    const uint32_t resident = aheadConvResident(L.bytes), keep = (perUnit < resident) ? (uint32_t)perUnit : resident;
    for(uint32_t depth = (inputs / 16 * 4 < AHEAD_CONV_MOST) ? inputs / 16 * 4 : AHEAD_CONV_MOST; L.fits && depth != 0; depth -= 4) {
        const size_t bytes = aheadConvBytes(inputs, (L.rowsPerBlock + kh - 1) * L.rowPitch, depth);
        if(aheadConvResident(bytes) >= keep) {
            L.listDepth = depth; L.bytes = bytes;
            break;
        }
    }
    return L;
}

// How many inputs of a pixel may have a spike in a step for its sum to be made one by one, by how many of a patch's words have spikes and how many those have (of
// the steps of a launch).  0: sums are products throughout.  (The line's figures: aheadConvKernel.)
constexpr uint32_t aheadConvMost(uint32_t depth, uint32_t inputs, uint32_t steps, uint32_t active, uint32_t spikes, uint32_t words)
{
    const uint64_t all = words, spikesOfAll = (uint64_t)spikes * inputs;
    const bool few = (32u * spikesOfAll <= 13ull * depth * steps * all), worth = (8ull * inputs * active > all * (4u * steps + 25u * ((inputs + 31u) / 32u)) + spikesOfAll);
    return (few && worth) ? depth : 0u;
}
}
