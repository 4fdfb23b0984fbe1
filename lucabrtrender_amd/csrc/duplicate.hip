// Duplication: one (tile, depth) key per tile a splat's footprint touches,
// written at the splat's offset from the exclusive scan of the touched counts.
// Repeats the projection's exact tile test, as the reference's splatEmit does
// (shaders/lrt/splat/splat_emit.slang:17-50), so each splat writes exactly the
// count it was given.
//
// Keys are 64-bit: tile id in the high word, the view depth's float bits in
// the low word (positive floats order as their bits). Values are slots. The
// pairs leave this kernel in slot order, which is what makes one stable sort on
// (tile, depth >> 7) give each tile its splats in the reference's order:
// depth key first, slot on ties.
//
// For a render whose gradients will be asked for, the value is instead the
// pair's own index in this slot-major order (and its slot goes to pairSlot):
// after the sort each pair then knows where its splat's run of pairs lies, so
// per-pair gradients written there sum per splat over contiguous runs.
//
// A frame of many pairs a slot duplicates its drawn slots in depth order
// instead (duplicateOrdered): the keys are then the tiles alone, u16 where the
// frame has no more than 65,536, and one stable sort by tile is enough.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "splat_math.h"

namespace lrt::kern {
namespace {

using namespace lrt::dev;

constexpr uint32_t kBlock = 256;

// Writes pair `at` of slot s, or counts it as past the capacity.
template <bool EMIT_INDEX, typename Key>
__device__ __forceinline__ void emitPair(uint32_t at, uint32_t index, Key key, uint32_t s, Key* __restrict__ keys,
                                         uint32_t* __restrict__ values, uint32_t* __restrict__ pairSlot,
                                         uint32_t capacity, uint32_t* __restrict__ overflow) {
    if (at < capacity) {
        keys[at] = key;
        if constexpr (EMIT_INDEX) {
            values[at] = index;
            if constexpr (sizeof(Key) == 8) pairSlot[index] = s;   // (else fillPairSlots', in slot order)
        } else {
            values[at] = s;
        }
    } else {
        atomicAdd(overflow, 1u);
    }
}

// The wave's slots' pairs: keys (tileBase + tile) << 32 | bits(view z) in the
// frame of width x height with tilesX tiles a row, each slot's in the
// row-major order of its tile rectangle, stopping at the count the projection
// gave. Every lane's rectangle is one run of a wave-wide candidate list
// (countTouchedTilesWave); a round tests 64 consecutive candidates, and a
// touched tile's pair goes to its slot's offset plus the slot's pairs so far
// plus its rank among this round's touched tiles of the same slot -- the place
// the one-lane row-major walk gives it. Every lane of the wave must take part
// (a lane with nothing to write passes expected 0). PER_VIEW: the frame sizes
// differ across lanes and travel with each candidate. With depthRange
// non-null, a slot whose depth key (bits(z) >> 7) lies outside
// [depthRange[0], depthRange[1]] is counted in *outOfRange.
// `first` is the place of the slot's first pair. Key u64: the keys as above. A
// narrower Key: the tile alone, for slots that come in depth order (not
// consecutive), with EMIT_INDEX each with the slot-order index of its first
// pair (`firstIndex`).
template <bool EMIT_INDEX, bool PER_VIEW, typename Key>
__device__ __forceinline__ void duplicateWave(uint32_t s, uint32_t expected, uint32_t first, uint32_t firstIndex,
                                              uint32_t width, uint32_t height,
                                              uint32_t tilesX, uint32_t tileShift, uint32_t tileBase,
                                              const float4* __restrict__ proj,
                                              const uint2* __restrict__ rects,
                                              Key* __restrict__ keys, uint32_t* __restrict__ values,
                                              uint32_t* __restrict__ pairSlot, uint32_t capacity,
                                              uint32_t* __restrict__ overflow,
                                              const uint32_t* __restrict__ depthRange,
                                              uint32_t* __restrict__ outOfRange) {
    const uint32_t lane = __lane_id();
    constexpr bool kOrdered = sizeof(Key) < 8;
    uint32_t x0 = 0, y0 = 0, w = 1, area = 0;
    float4 screen = make_float4(0.0f, 0.0f, 0.0f, 0.0f), conic = screen;
    if (expected != 0) {
        screen = proj[static_cast<uint64_t>(s) * 3];
        conic = proj[static_cast<uint64_t>(s) * 3 + 1];
        const uint2 rc = rects[s];
        x0 = rc.x & 0xFFFFu, y0 = rc.x >> 16;
        w = (rc.y & 0xFFFFu) - x0 + 1u;
        area = w * ((rc.y >> 16) - y0 + 1u);
    }
    const uint32_t depthBits = floatToBits(screen.z);
    if (depthRange != nullptr && expected != 0) {
        const uint32_t depthKey = (depthBits & 0x7FFFFFFFu) >> 7;
        if (depthKey < depthRange[0] || depthKey > depthRange[1]) atomicAdd(outOfRange, 1u);
    }
    const WaveTiles wt = waveTiles(area);
    const bool exact = wt.total >= (1u << 20);
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t slotOfLane0 = s - lane;   // in slot order the wave's slots are consecutive
    uint32_t written = 0;                    // this lane's slot's pairs so far
    for (uint32_t base = 0; base < wt.total; base += 64) {
        const uint32_t cand = base + lane;
        const uint32_t o = ownerOf(wt.incl, cand);
        const uint32_t oStart = shflU(wt.start, o), oW = shflU(w, o), ox0 = shflU(x0, o), oy0 = shflU(y0, o);
        const float ocx = shflF(screen.x, o), ocy = shflF(screen.y, o), ocut = shflF(screen.w, o);
        const float oa = shflF(conic.x, o), ob = shflF(conic.y, o), oc = shflF(conic.z, o);
        uint32_t ow = width, oh = height, oTilesX = tilesX, oBase = tileBase;
        if constexpr (PER_VIEW) {
            ow = shflU(width, o);
            oh = shflU(height, o);
            oTilesX = shflU(tilesX, o);
            oBase = shflU(tileBase, o);
        }
        const uint32_t oFirst = shflU(first, o), oExpected = shflU(expected, o), oWritten = shflU(written, o);
        uint32_t oDepth = 0, oSlot = slotOfLane0 + o, oIndex = oFirst;
        if constexpr (kOrdered) {
            oSlot = shflU(s, o);
            if constexpr (EMIT_INDEX) oIndex = shflU(firstIndex, o);
        } else {
            oDepth = shflU(depthBits, o);
        }
        bool hit = false;
        uint32_t tx = 0, ty = 0;
        if (cand < wt.total) {
            uint32_t row, col;
            rowColumn(cand - oStart, oW, exact, row, col);
            tx = ox0 + col;
            ty = oy0 + row;
            hit = tileTouched(ow, oh, ocx, ocy, oa, ob, oc, ocut, tx, ty, tileShift);
        }
        const uint64_t vote = __ballot(hit);
        if (hit) {
            // The owner's run begins at bit runLo of this round (at or below this lane).
            const uint32_t runLo = oStart > base ? oStart - base : 0u;
            const uint64_t sameRunBelow = below & ~((1ull << runLo) - 1ull);
            const uint32_t place = oWritten + static_cast<uint32_t>(__popcll(vote & sameRunBelow));
            if (place < oExpected) {
                const uint32_t tile = oBase + ty * oTilesX + tx;
                Key key;
                if constexpr (kOrdered) {
                    key = static_cast<Key>(tile);
                } else {
                    key = (static_cast<uint64_t>(tile) << 32) | oDepth;
                }
                emitPair<EMIT_INDEX>(oFirst + place, oIndex + place, key, oSlot, keys, values, pairSlot, capacity,
                                     overflow);
            }
        }
        written += static_cast<uint32_t>(__popcll(vote & runMask(wt.start, wt.area, base)));
    }
}

template <bool EMIT_INDEX>
__global__ __launch_bounds__(kBlock) void duplicateKernel(FrameParams f, uint32_t slots,
                                                          const float4* __restrict__ proj,
                                                          const uint2* __restrict__ rects,
                                                          const uint32_t* __restrict__ touched,
                                                          const uint32_t* __restrict__ offsets,
                                                          uint64_t* __restrict__ keys,
                                                          uint32_t* __restrict__ values,
                                                          uint32_t* __restrict__ pairSlot, uint32_t capacity,
                                                          uint32_t* __restrict__ overflow,
                                                          const uint32_t* __restrict__ depthRange,
                                                          uint32_t* __restrict__ outOfRange) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t expected = s < slots ? touched[s] : 0u;   // every lane stays for the wave's walk
    duplicateWave<EMIT_INDEX, false>(s, expected, expected != 0 ? offsets[s] : 0u, 0u, f.width, f.height, f.tilesX,
                                     f.tileShift, 0u, proj, rects, keys, values, pairSlot, capacity, overflow,
                                     depthRange, outOfRange);
}

// pairSlot[i] = s for every pair i of slot s in slot order: a wave's 64 slots'
// pairs are one range, written 64 a round, each place's slot found among the
// lanes' ends (the depth-ordered duplication would write each slot's few words
// to a place of their own).
__global__ __launch_bounds__(kBlock) void fillPairSlotsKernel(uint32_t slots, const uint32_t* __restrict__ touched,
                                                              const uint32_t* __restrict__ offsets,
                                                              uint32_t* __restrict__ pairSlot, uint32_t capacity) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t lane = __lane_id();
    const WaveTiles wt = waveTiles(s < slots ? touched[s] : 0u);
    if (wt.total == 0) return;   // uniform across the wave
    const uint32_t first = offsets[s - lane];   // lane 0's slot: every later lane's pairs follow
    for (uint32_t base = 0; base < wt.total; base += 64) {
        const uint32_t o = ownerOf(wt.incl, base + lane);
        const uint32_t at = first + base + lane;
        if (base + lane < wt.total && at < capacity) pairSlot[at] = s - lane + o;
    }
}

// The drawn slots in depth order: thread j takes order[j].
template <bool EMIT_INDEX, typename Key>
__global__ __launch_bounds__(kBlock) void duplicateOrderedKernel(
    FrameParams f, uint32_t slots, uint32_t count, const uint32_t* __restrict__ order, const float4* __restrict__ proj,
    const uint2* __restrict__ rects, const uint32_t* __restrict__ touched, const uint32_t* __restrict__ offsets,
    const uint32_t* __restrict__ slotOffsets, Key* __restrict__ keys, uint32_t* __restrict__ values,
    uint32_t capacity, uint32_t* __restrict__ overflow,
    const uint32_t* __restrict__ depthRange, uint32_t* __restrict__ outOfRange) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    uint32_t s = j < count ? order[j] : slots;
    uint32_t expected = 0, first = 0, firstIndex = 0;
    if (s < slots) {
        expected = touched[s];
        first = offsets[j];
        if constexpr (EMIT_INDEX) firstIndex = slotOffsets[s];
    }
    duplicateWave<EMIT_INDEX, false>(s, expected, first, firstIndex, f.width, f.height, f.tilesX, f.tileShift, 0u, proj,
                                     rects, keys, values, nullptr, capacity, overflow, depthRange, outOfRange);
}

// A batch of views: slot s belongs to view s / splatsPerView.
template <bool EMIT_INDEX>
__global__ __launch_bounds__(kBlock) void duplicateViewsKernel(const ViewInfo* __restrict__ views,
                                                               uint32_t splatsPerView, uint32_t tileShift, uint32_t slots,
                                                               const float4* __restrict__ proj,
                                                               const uint2* __restrict__ rects,
                                                               const uint32_t* __restrict__ touched,
                                                               const uint32_t* __restrict__ offsets,
                                                               uint64_t* __restrict__ keys,
                                                               uint32_t* __restrict__ values,
                                                               uint32_t* __restrict__ pairSlot, uint32_t capacity,
                                                               uint32_t* __restrict__ overflow,
                                                               uint32_t* __restrict__ outOfRange) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t expected = s < slots ? touched[s] : 0u;   // every lane stays for the wave's walk
    uint32_t width = 0, height = 0, tilesX = 0, tileBase = 0;
    const uint32_t* depthRange = nullptr;
    if (expected != 0) {
        const ViewInfo& v = views[s / splatsPerView];
        width = v.width;
        height = v.height;
        tilesX = v.tilesX;
        tileBase = v.tileBase;
        if (outOfRange != nullptr) depthRange = &v.depthLo;   // depthLo, depthHi
    }
    duplicateWave<EMIT_INDEX, true>(s, expected, expected != 0 ? offsets[s] : 0u,
                                    expected != 0 ? offsets[s] : 0u, width, height, tilesX, tileShift, tileBase, proj,
                                    rects, keys, values, pairSlot, capacity, overflow, depthRange, outOfRange);
}

}   // namespace

void duplicate(const FrameParams& f, uint32_t slots, const float4* proj, const uint2* rects,
               const uint32_t* touched, const uint32_t* offsets, uint64_t* keys, uint32_t* values,
               uint32_t* pairSlot, uint32_t capacity, uint32_t* overflow, hipStream_t stream,
               const uint32_t* depthRange, uint32_t* outOfRange) {
    if (slots == 0) return;
    const uint32_t blocks = (slots + kBlock - 1) / kBlock;
    if (pairSlot != nullptr) {
        duplicateKernel<true><<<blocks, kBlock, 0, stream>>>(f, slots, proj, rects, touched, offsets, keys, values,
                                                             pairSlot, capacity, overflow, depthRange, outOfRange);
    } else {
        duplicateKernel<false><<<blocks, kBlock, 0, stream>>>(f, slots, proj, rects, touched, offsets, keys, values,
                                                              nullptr, capacity, overflow, depthRange, outOfRange);
    }
}

template <typename Key>
void duplicateOrdered(const FrameParams& f, uint32_t slots, uint32_t count, const uint32_t* order, const float4* proj,
                      const uint2* rects, const uint32_t* touched, const uint32_t* offsets,
                      const uint32_t* slotOffsets, Key* keys, uint32_t* values, uint32_t* pairSlot, uint32_t capacity,
                      uint32_t* overflow, hipStream_t stream, const uint32_t* depthRange, uint32_t* outOfRange) {
    if (count == 0) return;
    const uint32_t blocks = (count + kBlock - 1) / kBlock;
    if (pairSlot != nullptr) {
        fillPairSlotsKernel<<<(slots + kBlock - 1) / kBlock, kBlock, 0, stream>>>(slots, touched, slotOffsets,
                                                                                 pairSlot, capacity);
        duplicateOrderedKernel<true, Key><<<blocks, kBlock, 0, stream>>>(f, slots, count, order, proj, rects, touched,
                                                                        offsets, slotOffsets, keys, values, capacity,
                                                                        overflow, depthRange, outOfRange);
    } else {
        duplicateOrderedKernel<false, Key><<<blocks, kBlock, 0, stream>>>(f, slots, count, order, proj, rects, touched,
                                                                         offsets, nullptr, keys, values, capacity,
                                                                         overflow, depthRange, outOfRange);
    }
}
template void duplicateOrdered<uint16_t>(const FrameParams&, uint32_t, uint32_t, const uint32_t*, const float4*,
                                         const uint2*, const uint32_t*, const uint32_t*, const uint32_t*, uint16_t*,
                                         uint32_t*, uint32_t*, uint32_t, uint32_t*, hipStream_t, const uint32_t*,
                                         uint32_t*);
template void duplicateOrdered<uint32_t>(const FrameParams&, uint32_t, uint32_t, const uint32_t*, const float4*,
                                         const uint2*, const uint32_t*, const uint32_t*, const uint32_t*, uint32_t*,
                                         uint32_t*, uint32_t*, uint32_t, uint32_t*, hipStream_t, const uint32_t*,
                                         uint32_t*);

void duplicateViews(const ViewInfo* views, uint32_t splatsPerView, uint32_t tileShift, uint32_t slots,
                    const float4* proj,
                    const uint2* rects, const uint32_t* touched, const uint32_t* offsets, uint64_t* keys,
                    uint32_t* values, uint32_t* pairSlot, uint32_t capacity, uint32_t* overflow,
                    uint32_t* outOfRange, hipStream_t stream) {
    if (slots == 0 || splatsPerView == 0) return;
    const uint32_t blocks = (slots + kBlock - 1) / kBlock;
    if (pairSlot != nullptr) {
        duplicateViewsKernel<true><<<blocks, kBlock, 0, stream>>>(views, splatsPerView, tileShift, slots, proj, rects,
                                                                  touched,
                                                                  offsets, keys, values, pairSlot, capacity, overflow,
                                                                  outOfRange);
    } else {
        duplicateViewsKernel<false><<<blocks, kBlock, 0, stream>>>(views, splatsPerView, tileShift, slots, proj, rects,
                                                                   touched,
                                                                   offsets, keys, values, nullptr, capacity, overflow,
                                                                   outOfRange);
    }
}

}   // namespace lrt::kern
