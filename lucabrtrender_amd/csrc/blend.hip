// Blend: one workgroup per 16x16 block of a tile (a 16x16 tile is one, a 32x32
// tile four; an 8x8 tile is a block of its own), one wave per 8x8 quadrant of
// it, one lane per pixel. The workgroup walks its tile's sorted pairs front to
// back in rounds of a pair a lane:
//   1. each lane stages one pair (its record gathered a round ahead, so the
//      load is in flight while the last round is walked): it tests the pair
//      against each quadrant's pixel-centre box with a conservative bound on
//      the Gaussian's power (quadrantReach), puts the record into the LDS and
//      its place into the list of every quadrant it can reach (ballot +
//      popcount), in pair order;
//   2. after a barrier each wave walks its quadrant's list, four records a
//      group, and leaves once its 64 pixels are opaque. Records and lists hold
//      two rounds, so one barrier a round is enough.
// A tile's four quadrants share one gather and one staging of its pairs. With a
// wave of its own for each quadrant, each gathered and tested all of them: 26.9M
// cache accesses a launch against 7.4M on 3M splats at 1920x1080.
// A record's Gaussian is expanded about the quadrant's centre and scaled to the
// exponent's base 2, log2(opacity) added: at a pixel (u, v) from the
// centre q = A u^2 + B u v + C v^2 + D u + E v + F, the pixel is inside the
// cutoff and above the alpha floor when q >= the record's bound, and alpha =
// min(0.99, 2^q). q differs from the direct form's
// scaled power by float rounding only (below 2e-4 on footprints from a quarter
// pixel to 300 pixels wide, centres up to 3.5 sigma outside the quadrant).
//
// What bounds it: vector issue in the walk (busy 61% of a launch on 3M splats at
// 1920x1080, the matrix cores 12%; 67 vector instructions a group of four
// records, staging included), and between its instructions the chain through T,
// the rounds' gathers and barriers and the launch's last tiles. A wave a quadrant
// with form and colours on FMAs, the records read from the LDS by broadcast,
// issued 84.2M vector instructions a launch there against 57.0M, and 10.7M LDS
// instructions against 5.7M. Blend time, that form against this one: 3M clustered
// splats at 1920x1080 232 against 194 us, with 1M discs 217 against 179; 2M
// splats in 64 views 4.93 against 4.10 ms; 1M splats at 1571x877 with the
// threshold depth 95 against 75 us. Broadcasting the records by DPP operands
// instead took 198 us where six matrix products for the form took 178.
//
// Per pixel it is the reference's splatBlend walk (shaders/lrt/splat/
// splat_blend.slang:23-108, splat-only entry :110-114): skip past the cutoff,
// alpha = min(0.99, opacity * exp(-power / 2)), skip below 1/255, accumulate
// with the transmittance, stop below 1e-4, then linearise rgb / coverage. The
// Gaussian's exponent runs on the hardware exp2 and the quadratic form on
// matrix FMAs in f32; both move the result by a few ulps, which the image
// tolerances cover.
//
// The composite walk (splatBlendComposite, :116-120) is the same kernel
// instantiated with COMPOSITE: a disc record (colour.w 1) that reaches a pixel
// ends its walk and lies behind what it blended; a pixel with an under-layer
// depth above 0 ends its walk at the first pair of its tile at or behind that
// depth. That first pair may be one the quadrant's list dropped, so each staged
// record carries the largest view z of every pair up to it (a wave max-scan at
// staging, the waves and rounds before added when it is walked), and the walk
// tests that instead of the record's own z.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "splat_math.h"

namespace lrt::kern {
namespace {

using namespace lrt::dev;

constexpr uint32_t kLanes = 64;          // one wave: an 8x8 quadrant
constexpr uint32_t kGroup = 4;           // list records walked per step
constexpr float kAlphaMax = 0.99f;       // a splat's alpha at most (splat_blend.slang:66)
constexpr float kExpScale = -0.72134752044448170368f;   // -log2(e) / 2
constexpr float kLog2Floor = -7.99435343685885793775f;   // log2(1 / 255): alpha's floor

// The sRGB decode (reference color.slang:7-10) on the hardware log2 and exp2,
// the division by the coverage a reciprocal: a few ulps, as the walk's own
// exponent (the blend's images match the oracle within the image tolerances,
// not bit for bit; the projection, counts and keys stay exact).
__device__ __forceinline__ float srgbToLinearFast(float c) {
    c = fmaxS(c, 0.0f);
    return c <= 0.04045f ? c * (1.0f / 12.92f)
                         : __builtin_amdgcn_exp2f(2.4f * __builtin_amdgcn_logf((c + 0.055f) * (1.0f / 1.055f)));
}

// The finished pixel: linearise rgb / coverage, the background behind, the
// depth (reference splat_blend.slang:89-107, splat-only).
__device__ __forceinline__ void finishPixel(const FrameParams& f, uint32_t px, uint32_t py, float r, float g, float b,
                                            float t, float depthSum, float depthAt, uint32_t last,
                                            float4* __restrict__ colour, float* __restrict__ depth,
                                            uint32_t* __restrict__ lastCount, float* __restrict__ finalT,
                                            float4* __restrict__ accum) {
    const float coverage = 1.0f - t;
    if (accum != nullptr) accum[py * f.width + px] = make_float4(r, g, b, depthSum);
    if (f.linearise && coverage > 1e-6f) {
        const float inv = __builtin_amdgcn_rcpf(coverage);
        r = srgbToLinearFast(r * inv) * coverage;
        g = srgbToLinearFast(g * inv) * coverage;
        b = srgbToLinearFast(b * inv) * coverage;
    }
    const uint32_t at = py * f.width + px;
    colour[at] = make_float4(r + t * f.bg[0], g + t * f.bg[1], b + t * f.bg[2], coverage + t * f.bg[3]);
    if (depth != nullptr) {
        depth[at] = f.depthMode == 0 ? (coverage > 1e-6f ? depthSum / coverage : 0.0f) : fmaxS(depthAt, 0.0f);
    }
    if (lastCount != nullptr) lastCount[at] = last;
    if (finalT != nullptr) finalT[at] = t;
}

// The finished pixel of the composite walk (reference splat_blend.slang:83-107):
// without a disc, the under-layer lies behind; whatever lies behind is
// composited under the linearised splats and weighs in the depth with the
// transmittance left.
__device__ __forceinline__ void finishComposite(const FrameParams& f, uint32_t at, float r, float g, float b, float t,
                                                float depthSum, float depthAt, bool opaqueHit, float4 opaque,
                                                float opaqueZ, bool underHit, const float4* __restrict__ underColour,
                                                float underZ, float4* __restrict__ colour, float* __restrict__ depth) {
    if (!opaqueHit && underHit) {
        opaqueHit = true;
        opaque = underColour[at];
        opaqueZ = underZ;
    }
    const float coverage = 1.0f - t;
    if (f.linearise && coverage > 1e-6f) {
        const float inv = __builtin_amdgcn_rcpf(coverage);
        r = srgbToLinearFast(r * inv) * coverage;
        g = srgbToLinearFast(g * inv) * coverage;
        b = srgbToLinearFast(b * inv) * coverage;
    }
    float4 behind = make_float4(f.bg[0], f.bg[1], f.bg[2], f.bg[3]);
    if (opaqueHit) {
        behind = opaque;
        depthSum = depthSum + t * opaqueZ;
        if (depthAt < 0.0f) depthAt = opaqueZ;
    }
    const float total = opaqueHit ? 1.0f : coverage;
    colour[at] = make_float4(r + t * behind.x, g + t * behind.y, b + t * behind.z, coverage + t * behind.w);
    if (depth != nullptr) {
        depth[at] = f.depthMode == 0 ? (total > 1e-6f ? depthSum / total : 0.0f) : fmaxS(depthAt, 0.0f);
    }
}

constexpr uint32_t kNoSlot = 0xFFFFFFFFu;   // no pair; a task that finishes its tile's pixels itself

// One pair's projected record, or an empty one (cutoff -1) past the range.
struct Staged {
    float4 screen;   // centre.xy, view z, cutoff
    float4 conic;    // a, b, c, alpha
    float4 col;      // rgb, 0
};

// Orders a wave's own LDS writes and reads: its lanes run together, so only
// the compiler has to keep them in order.
__device__ __forceinline__ void waveSync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// Inclusive max-scan over the wave's lanes: within rows of sixteen by row
// shifts, then row 0 into row 1 and row 2 into row 3 (row_bcast:15), then rows
// 0-1 into rows 2-3 (row_bcast:31); a lane with no source reads the least.
template <int CTRL, int ROWS>
__device__ __forceinline__ float maxWith(float v) {
    const int least = __float_as_int(-3.4e38f);
    return __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(least, __float_as_int(v), CTRL, ROWS, 0xF, false)));
}
__device__ __forceinline__ float waveMaxScan(float v) {
    v = maxWith<0x111, 0xF>(v);   // row_shr:1, 2, 4, 8
    v = maxWith<0x112, 0xF>(v);
    v = maxWith<0x114, 0xF>(v);
    v = maxWith<0x118, 0xF>(v);
    v = maxWith<0x142, 0xA>(v);
    return maxWith<0x143, 0xC>(v);
}

__device__ __forceinline__ Staged gather(const float4* __restrict__ proj, uint32_t slot, uint32_t slots) {
    Staged s{make_float4(0.0f, 0.0f, 0.0f, -1.0f), make_float4(0.0f, 0.0f, 0.0f, 0.0f),
             make_float4(0.0f, 0.0f, 0.0f, 0.0f)};
    if (slot < slots) {
        const uint64_t s3 = static_cast<uint64_t>(slot) * 3;
        s.screen = proj[s3];
        s.conic = proj[s3 + 1];
        s.col = proj[s3 + 2];
    }
    return s;
}

// A block's LDS: the workgroup's waves each take one 8x8 quadrant of its
// block (four waves a 16x16 block; one wave an 8x8 one), and all of them stage
// the block's pairs, a round of a pair a lane at a time, two rounds' worth so
// that one barrier a round is enough (a wave may stage the next round while
// another still walks this one).
template <uint32_t WAVES, bool COMPOSITE>
struct BlendShared {
    static constexpr uint32_t kRound = WAVES * kLanes;
    // The round's records, in pair order, the conic scaled to base 2:
    float4 at[2][kRound];       // centre.xy, A, B
    float4 shape[2][kRound];    // C, what F adds to the form at the centre, the test's bound, 0
    float4 colour[2][kRound];   // rgb, view z
    // Composite: the largest view z of the record's wave's pairs up to it, kept or not, and each wave's.
    float reach[2][COMPOSITE ? kRound : 1];
    float most[2][WAVES];
    // Quadrant q's records among those source wave w staged: lanes in order, and how many.
    uint8_t list[2][WAVES][kRound];
    uint32_t count[2][WAVES][WAVES];
    uint32_t done[2][WAVES];    // the wave's pixels all stopped before this round
    // A wave's own: of the chunk it walks, four records a vector, D, E, F, the
    // test's bound (and the reach).
    float4 chunk[WAVES][4][kLanes / 4];
    float4 chunkReach[WAVES][COMPOSITE ? kLanes / 4 : 1];
};

// A pixel's walk so far: premultiplied rgb, transmittance, depth sum, the
// threshold depth (-1: not reached), the place of the last contributor, and
// whether it still walks.
struct WalkState {
    float r, g, b, t, depthSum, depthAt;
    uint32_t last;
    bool active;
};

// What a walk leaves (MODE): kFinish writes the finished pixel; kPartial
// writes the walk's state as it stands at the range's end (a segment of a
// split tile, walked from an empty state) to partialA/partialB[lane];
// kResume starts from *state (its active lanes) and leaves the state there.
constexpr uint32_t kFinish = 0, kPartial = 1, kResume = 2;

// A tile of side 2^tileShift holds 2^quadBits 8x8 quadrants (1, 4 or 16) and
// 2^blockBits blocks (of four quadrants, but an 8-pixel tile's one), numbered
// row-major inside it.
__host__ __device__ __forceinline__ uint32_t quadBits(uint32_t tileShift) { return 2u * (tileShift - 3u); }
__host__ __device__ __forceinline__ uint32_t blockBits(uint32_t tileShift) {
    return tileShift <= 4u ? 0u : 2u * (tileShift - 4u);
}

// The first pixel of part `part` of tile `tile` of the frame f, its parts
// 2^partShift pixels square.
__device__ __forceinline__ uint2 partOrigin(const FrameParams& f, uint32_t tile, uint32_t part, uint32_t partShift) {
    const uint32_t side = f.tileShift - partShift;
    return make_uint2(((tile % f.tilesX) << f.tileShift) + ((part & ((1u << side) - 1u)) << partShift),
                      ((tile / f.tilesX) << f.tileShift) + ((part >> side) << partShift));
}

using Vec4 = float __attribute__((ext_vector_type(4)));

// A pixel's walk while it runs: accum holds rgb and the depth sum. The pixel
// walks while t >= kTMin; composite: a pixel that something behind stops leaves
// its T in tStopped and t 0. lastIn, depthIn and opaqueIn: a record's place in
// the chunk at hand (-1: none yet).
struct WalkLane {
    Vec4 accum;
    float t, tStopped;
    float depthAt;   // the depth is found once 1 - T is at least this; infinite once found
    int32_t lastIn, depthIn, opaqueIn;
};
constexpr float kTMin = 1e-4f;
// Waves a SIMD the register allocation leaves room for: at two and more the
// matrix results stay in the vector registers (no copies from accumulators).
constexpr uint32_t kWavesPerSimd = 4;

// The form of records 4 G .. 4 G + 3 of sixteen at the lane's own pixel:
// q = u (A u + (B v + D)) + (v (C v + E) + F), each step a fused multiply-add.
//
// The walk's contractions run on the matrix cores, in f32, as sixteen 4x4
// blocks of four lanes a block (v_mfma_f32_4x4x1, one block's lanes of A given
// to every block): a product and a sum rounded once, bit for bit the fused
// multiply-add. The form's three products of a coefficient and the pixel's u or
// v: rows of records times columns of pixels; lane l < 16 of `form` holds record
// l's A, B and C, block G's four lanes are records 4 G .. 4 G + 3, q[k] lands in
// the lane of its pixel, and D, E and F (four records' a vector, one LDS read
// each) start the sums. The two outer steps multiply by a sum of the pixel's
// own and stay on the VALU. The colours: rows of channels times columns of
// pixels, one product a record, summed into the lane's own accum; lane l of
// `colour`: channel l & 3 of record l / 4. What stays on the VALU besides is
// what is no contraction: the exponential, the tests and T.
//
// Every step rounds as the walk of one record after the other on FMAs does, so
// a pair at its cutoff or at the alpha floor falls on the same side. (The six
// terms as one sum of six products, all on the matrix cores, rounds otherwise:
// about one pixel-pair in ten million fell the other way, a whole contribution
// each. Frames took 1 to 2 % less time with it.)
template <uint32_t G>
__device__ __forceinline__ Vec4 formOf(const float form[3], float u, float v, const float4 (*chunk)[kLanes / 4],
                                       uint32_t at) {
    const float4 d = chunk[0][at + G], e = chunk[1][at + G], f = chunk[2][at + G];
    Vec4 x = {d.x, d.y, d.z, d.w}, y = {e.x, e.y, e.z, e.w};
    x = __builtin_amdgcn_mfma_f32_4x4x1f32(form[1], v, x, 4, G, 0);
    y = __builtin_amdgcn_mfma_f32_4x4x1f32(form[2], v, y, 4, G, 0);
    x = __builtin_amdgcn_mfma_f32_4x4x1f32(form[0], u, x, 4, G, 0);
    const float f4[4] = {f.x, f.y, f.z, f.w};
    Vec4 q;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) q[k] = __builtin_fmaf(u, x[k], __builtin_fmaf(v, y[k], f4[k]));
    return q;
}

// One record's colour into the pixel's sums.
template <uint32_t R>
__device__ __forceinline__ Vec4 addColour(float colour, float weight, Vec4 accum) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(colour, weight, accum, 4, R, 0);
}

// One group of kGroup records, 4 G .. 4 G + 3 of the sixteen at hand, with form
// q. A wave's records are one serial chain through T, and a launch cannot end
// before its longest tile's chain, so the chain is kept short: the four
// weights are taken as if no pixel stopped among the first three records (a
// product and a difference a record on the chain), and a group in which one does is
// taken again with the test between the records. Both ways do the same
// arithmetic for a pixel that does not stop.
template <uint32_t DEPTH_MODE, bool COMPOSITE, bool TRACK, uint32_t G>
__device__ __forceinline__ void walkGroup(WalkLane& w, Vec4 q, float colour, float4 bound4, float4 reach4,
                                          float stopZ, uint64_t discs, int32_t first) {
    constexpr uint32_t R0 = G * kGroup;
    const float bound[4] = {bound4.x, bound4.y, bound4.z, bound4.w};
    bool passes[4];   // inside the cutoff and above the alpha floor
    bool inside[4];   // composite: inside the cutoff
    float alpha[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const float power2 = __builtin_amdgcn_exp2f(q[k]);
        if constexpr (COMPOSITE) {
            const float a = bound[k] * power2;
            inside[k] = q[k] >= 0.0f;
            passes[k] = inside[k] & (a >= 1.0f / 255.0f);
            alpha[k] = passes[k] ? __builtin_fminf(kAlphaMax, a) : 0.0f;
        } else {
            passes[k] = q[k] >= bound[k];
            alpha[k] = passes[k] ? __builtin_fminf(kAlphaMax, power2) : 0.0f;
        }
    }
    float weight[4];
    if constexpr (COMPOSITE) {
        // A group with a disc, or that an under-layer ends in, goes record by
        // record. The reach grows along the list (padding has the last one's),
        // so a group's last says whether one of it ends a pixel's walk.
        const float reach[4] = {reach4.x, reach4.y, reach4.z, reach4.w};
        const bool ends = (w.t >= kTMin) & (reach[3] >= stopZ);
        const bool anyEnds = __ballot(ends) != 0;
        if (((discs >> R0) & 15u) != 0u || anyEnds) {
            const auto stop = [&](bool here) {
                w.tStopped = here ? w.t : w.tStopped;
                w.t = here ? 0.0f : w.t;
            };
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (anyEnds) stop((w.t >= kTMin) & (reach[k] >= stopZ));
                weight[k] = 0.0f;
                if (((discs >> (R0 + k)) & 1u) != 0u) {   // uniform: a disc that reaches the pixel ends its walk
                    const bool hit = (w.t >= kTMin) & inside[k];
                    w.opaqueIn = hit ? first + static_cast<int32_t>(R0 + k) : w.opaqueIn;
                    stop(hit);
                } else {
                    const bool here = w.t >= kTMin;
                    weight[k] = (here ? w.t : 0.0f) * alpha[k];
                    w.t = w.t - weight[k];
                    if constexpr (DEPTH_MODE == 1) {
                        const bool at = here & passes[k] & (1.0f - w.t >= w.depthAt);
                        w.depthIn = at ? first + static_cast<int32_t>(R0 + k) : w.depthIn;
                        w.depthAt = at ? __builtin_inff() : w.depthAt;
                    }
                }
            }
            w.accum = addColour<R0>(colour, weight[0], w.accum);
            w.accum = addColour<R0 + 1>(colour, weight[1], w.accum);
            w.accum = addColour<R0 + 2>(colour, weight[2], w.accum);
            w.accum = addColour<R0 + 3>(colour, weight[3], w.accum);
            return;
        }
    }
    const bool walks = w.t >= kTMin;
    float t[5];
    t[0] = walks ? w.t : 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        weight[k] = t[k] * alpha[k];
        t[k + 1] = t[k] - weight[k];   // T (1 - alpha)
    }
    bool ok[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) ok[k] = walks & passes[k];
    if (__ballot(walks & (t[3] < kTMin)) != 0) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool here = t[k] >= kTMin;
            ok[k] = here & passes[k];
            weight[k] = t[k] * (here ? alpha[k] : 0.0f);
            t[k + 1] = t[k] - weight[k];
        }
    }
    w.accum = addColour<R0>(colour, weight[0], w.accum);
    w.accum = addColour<R0 + 1>(colour, weight[1], w.accum);
    w.accum = addColour<R0 + 2>(colour, weight[2], w.accum);
    w.accum = addColour<R0 + 3>(colour, weight[3], w.accum);
    if constexpr (TRACK) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) w.lastIn = ok[k] ? first + static_cast<int32_t>(R0 + k) : w.lastIn;
    }
    if constexpr (DEPTH_MODE == 1) {
        // T only falls, so a group whose last T finds no pixel's depth holds
        // none; each pixel's is found once.
        if (__ballot(walks & (1.0f - t[4] >= w.depthAt)) != 0) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const bool at = ok[k] & (1.0f - t[k + 1] >= w.depthAt);
                w.depthIn = at ? first + static_cast<int32_t>(R0 + k) : w.depthIn;
                w.depthAt = at ? __builtin_inff() : w.depthAt;
            }
        }
    }
    w.t = walks ? t[4] : w.t;
}

// Up to sixteen records, whose A, B and C lanes 0 .. 15 hold and whose colours
// `colour` does (lane l: channel l & 3 of record l / 4), four a group in order,
// while there are records and the wave has a pixel that walks; the next group's
// form is computed, and its bounds read, while this one is blended. Returns the
// records walked.
template <uint32_t DEPTH_MODE, bool COMPOSITE, bool TRACK>
__device__ __forceinline__ uint32_t walkSixteen(WalkLane& w, uint32_t records, const float form[3], float colour,
                                                float u, float v, const float4 (*chunk)[kLanes / 4], uint32_t at,
                                                const float4* chunkReach, float stopZ, uint64_t discs,
                                                int32_t first) {
    uint32_t walked = 0;
    Vec4 q = formOf<0>(form, u, v, chunk, at);
    float4 bound = chunk[3][at];
    float4 reach = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (COMPOSITE) reach = chunkReach[0];
    const auto group = [&](auto g) -> bool {
        constexpr uint32_t G = decltype(g)::value;
        if (G * kGroup >= records) return false;
        Vec4 nextQ = q;
        float4 nextBound = bound, nextReach = reach;
        if constexpr (G + 1 < 16 / kGroup) {
            nextQ = formOf<G + 1>(form, u, v, chunk, at);
            nextBound = chunk[3][at + G + 1];
            if constexpr (COMPOSITE) nextReach = chunkReach[G + 1];
        }
        walkGroup<DEPTH_MODE, COMPOSITE, TRACK, G>(w, q, colour, bound, reach, stopZ, discs, first);
        q = nextQ;
        bound = nextBound;
        reach = nextReach;
        walked += kGroup;
        return __ballot(w.t >= kTMin) != 0;
    };
    (void)(group(std::integral_constant<uint32_t, 0>{}) && group(std::integral_constant<uint32_t, 1>{}) &&
           group(std::integral_constant<uint32_t, 2>{}) && group(std::integral_constant<uint32_t, 3>{}));
    return walked;
}

// The block of WAVES quadrants whose first pixel is `origin`, walking the pairs
// [range.x, range.y) of pairSlots (all of the tile's, or a segment of them;
// places count from tileStart); colour and depth are the frame's images,
// lastCount/finalT/accum its per-pixel state (each may be null). Every wave of
// the workgroup calls it; a workgroup that calls it again has a barrier in
// between (the LDS is the last call's until then).
template <uint32_t DEPTH_MODE, uint32_t WAVES, bool COMPOSITE, uint32_t MODE = kFinish, bool TRACK = true>
__device__ __forceinline__ void blendBlock(BlendShared<WAVES, COMPOSITE>& shared, const FrameParams& f, uint2 origin,
                                           uint2 range, uint32_t tileStart, uint32_t slots,
                                           const uint32_t* __restrict__ pairSlots, const float4* __restrict__ proj,
                                           const float4* __restrict__ underColour,
                                           const float* __restrict__ underDepth, float4* __restrict__ colour,
                                           float* __restrict__ depth, uint32_t* __restrict__ lastCount,
                                           float* __restrict__ finalT, float4* __restrict__ accum,
                                           WalkState* state = nullptr, float4* __restrict__ partialA = nullptr,
                                           float2* __restrict__ partialB = nullptr,
                                           uint32_t* __restrict__ walkSteps = nullptr,
                                           const uint32_t* __restrict__ slotOfPair = nullptr) {
    static_assert(!(COMPOSITE && MODE != kFinish), "a composite walk is not split");
    static_assert(WAVES == 1 || (WAVES == 4 && MODE == kFinish), "a quadrant, or the four of a 16x16 block");
    constexpr uint32_t kRound = WAVES * kLanes;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = WAVES == 1 ? 0u : threadIdx.x >> 6;
    // The block's quadrants: the pixel-centre box of each, empty past the frame's edge.
    float boxLo[WAVES][2], boxHi[WAVES][2];
    bool any[WAVES];
#pragma unroll
    for (uint32_t q = 0; q < WAVES; ++q) {
        const uint32_t x0 = origin.x + (q & 1u) * 8u, y0 = origin.y + (q >> 1) * 8u;
        any[q] = x0 < f.width && y0 < f.height;
        boxLo[q][0] = static_cast<float>(x0) + 0.5f;
        boxLo[q][1] = static_cast<float>(y0) + 0.5f;
        boxHi[q][0] = static_cast<float>(x0 + 8u < f.width ? x0 + 8u : f.width) - 0.5f;
        boxHi[q][1] = static_cast<float>(y0 + 8u < f.height ? y0 + 8u : f.height) - 0.5f;
    }
    const uint32_t px = origin.x + (wave & 1u) * 8u + (lane & 7u);
    const uint32_t py = origin.y + (wave >> 1) * 8u + (lane >> 3);
    const bool inside = px < f.width && py < f.height;
    // The pixel centre about the quadrant's centre, and that centre.
    const float pu = static_cast<float>(lane & 7u) - 3.5f;
    const float pv = static_cast<float>(lane >> 3) - 3.5f;
    const float xm = static_cast<float>(origin.x + (wave & 1u) * 8u) + 4.0f;
    const float ym = static_cast<float>(origin.y + (wave >> 1) * 8u) + 4.0f;
    const uint64_t below = (1ull << lane) - 1ull;

    // A training frame's sort carried pair indices: each pair's slot is read
    // through its index, a round ahead of its record.
    const auto valueAt = [&](uint32_t at) -> uint32_t { return at < range.y ? pairSlots[at] : kNoSlot; };
    const auto slotOf = [&](uint32_t v) -> uint32_t {
        return slotOfPair != nullptr && v != kNoSlot ? slotOfPair[v] : v;
    };
    const uint32_t mine = range.x + threadIdx.x;
    Staged staged = gather(proj, slotOf(valueAt(mine)), slots);
    uint32_t slotNext = slotOf(valueAt(mine + kRound));   // the next round's slot
    uint32_t valueNext = valueAt(mine + 2u * kRound);     // the value of the round after

    WalkLane w{{0.0f, 0.0f, 0.0f, 0.0f}, inside ? 1.0f : 0.0f, -1.0f, f.depthThreshold, -1, -1, -1};
    float depthAt = -1.0f;
    uint32_t last = 0;
    if constexpr (MODE == kResume) {
        w.accum = Vec4{state->r, state->g, state->b, state->depthSum};
        w.t = inside && state->active ? state->t : 0.0f;
        depthAt = state->depthAt;
        w.depthAt = depthAt < 0.0f ? w.depthAt : __builtin_inff();
        last = state->last;
    }
    // Composite: what ends the walk from behind. A pixel with an under depth
    // above 0 stops at the first pair at or behind it (whether or not that pair
    // reaches the pixel: the reference tests the depth first), a disc that
    // reaches the pixel stops it with its colour.
    const uint32_t at0 = py * f.width + px;
    float underZ = 0.0f;
    if constexpr (COMPOSITE) {
        if (underDepth != nullptr && inside) underZ = underDepth[at0];
    }
    const bool underHit = COMPOSITE && underZ > 0.0f;
    const float stopZ = underHit ? underZ : __builtin_inff();   // no finite depth reaches it
    bool opaqueHit = false;
    float oR = 0.0f, oG = 0.0f, oB = 0.0f, oZ = 0.0f;
    float zCarry = -3.4e38f;   // the largest view z of the rounds before
    uint32_t walked = 0;       // list records walked (kGroup a step)
    bool walks = __ballot(w.t >= kTMin) != 0;
    uint32_t buf = 0;
    for (uint32_t next = range.x; next < range.y; next += kRound, buf ^= 1u) {
        // 1. stage: each lane's record and which quadrants it can reach
        const uint32_t at = next + threadIdx.x;
        const uint32_t slot = wave * kLanes + lane;   // the record's place in the round
        uint32_t mask = 0;
        if (at < range.y) {
            const Staged& s = staged;
            const ReachConic rc = reachConic(s.conic.x, s.conic.y, s.conic.z);
#pragma unroll
            for (uint32_t q = 0; q < WAVES; ++q) {
                const bool reach = quadrantReach(rc, s.screen.w, boxLo[q][0] - s.screen.x, boxLo[q][1] - s.screen.y,
                                                 boxHi[q][0] - s.screen.x, boxHi[q][1] - s.screen.y);
                mask |= any[q] && reach ? 1u << q : 0u;
            }
        }
        if constexpr (COMPOSITE) {
            // inclusive max-scan of the wave's view z in pair order
            const float zr = waveMaxScan(at < range.y ? staged.screen.z : -3.4e38f);
            shared.reach[buf][slot] = zr;
            if (lane == kLanes - 1u) shared.most[buf][wave] = zr;
        }
        if (mask != 0) {
            const Staged& s = staged;
            const float scaledCut = kExpScale * s.screen.w;
            float base, bound;
            if constexpr (COMPOSITE) {
                // q = the form less the cutoff; alpha = o' 2^q, the bound o'. A
                // disc (colour.w 1) is marked by o' < 0: its alpha never passes.
                base = -scaledCut;
                bound = s.col.w > 0.5f ? -1.0f : s.conic.w * __builtin_amdgcn_exp2f(scaledCut);
            } else {
                // q = the form plus log2(opacity): alpha = 2^q directly, and both
                // tests (inside the cutoff, alpha >= 1/255) are q >= the bound
                base = __builtin_amdgcn_logf(s.conic.w);
                bound = fmaxS(base + scaledCut, kLog2Floor);
            }
            shared.at[buf][slot] = make_float4(s.screen.x, s.screen.y, kExpScale * s.conic.x,
                                               kExpScale * (s.conic.y + s.conic.y));
            shared.shape[buf][slot] = make_float4(kExpScale * s.conic.z, base, bound, 0.0f);
            shared.colour[buf][slot] = make_float4(s.col.x, s.col.y, s.col.z, s.screen.z);
        }
#pragma unroll
        for (uint32_t q = 0; q < WAVES; ++q) {
            const uint64_t vote = __ballot((mask >> q) & 1u);
            if ((mask >> q) & 1u) {
                shared.list[buf][q][wave * kLanes + static_cast<uint32_t>(__popcll(vote & below))] =
                    static_cast<uint8_t>(lane);
            }
            if (lane == q) shared.count[buf][q][wave] = static_cast<uint32_t>(__popcll(vote));
        }
        if (lane == 0) shared.done[buf][wave] = walks ? 0u : 1u;
        // 2. the next round's record, the slot of the one after and the value after that
        staged = gather(proj, slotNext, slots);
        slotNext = slotOf(valueNext);
        valueNext = valueAt(at + 3u * kRound);
        __syncthreads();
        if constexpr (WAVES > 1) {
            // Written before the barrier, read after it, written again only two
            // rounds on: every wave reads the same.
            uint32_t stopped = 1;
#pragma unroll
            for (uint32_t q = 0; q < WAVES; ++q) stopped &= shared.done[buf][q];
            if (stopped != 0) break;
        }
        float before[WAVES];   // composite: the largest view z ahead of each source wave's pairs
        if constexpr (COMPOSITE) {
#pragma unroll
            for (uint32_t q = 0; q < WAVES; ++q) {
                before[q] = zCarry;
                zCarry = fmaxS(zCarry, shared.most[buf][q]);
            }
        }
        if (!walks) {
            if constexpr (WAVES == 1) break;
            continue;
        }
        // 3. walk this quadrant's records, 64 a chunk: their coefficients and
        // colours a record a lane, for the matrix cores to hand round
        uint32_t start[WAVES + 1];
        start[0] = 0;
#pragma unroll
        for (uint32_t q = 0; q < WAVES; ++q) {
            start[q + 1] = start[q] + static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                                          static_cast<int>(shared.count[buf][wave][q])));
        }
        const uint32_t total = start[WAVES];
        for (uint32_t chunk = 0; chunk < total; chunk += kLanes) {
            const uint32_t k = chunk + lane;
            const bool real = k < total;
            const uint32_t kk = real ? k : total - 1u;
            uint32_t from = 0, first = 0;
#pragma unroll
            for (uint32_t q = 1; q < WAVES; ++q) {
                from = kk >= start[q] ? q : from;
                first = kk >= start[q] ? start[q] : first;
            }
            const uint32_t record = from * kLanes + shared.list[buf][wave][from * kLanes + (kk - first)];
            const float4 g0 = shared.at[buf][record];
            const float4 g1 = shared.shape[buf][record];
            // The form about the quadrant's centre; past the list, one that passes nothing.
            const float ux = g0.x - xm, vy = g0.y - ym;
            const float fa = g0.z, fb = g0.w, fc = g1.x;
            const float fd = -(2.0f * fa * ux + fb * vy), fe = -(2.0f * fc * vy + fb * ux);
            const float fbase = ux * (fa * ux + fb * vy) + fc * vy * vy;
            const float form[3] = {fa, fb, fc};
            reinterpret_cast<float*>(shared.chunk[wave][0])[lane] = fd;
            reinterpret_cast<float*>(shared.chunk[wave][1])[lane] = fe;
            reinterpret_cast<float*>(shared.chunk[wave][2])[lane] = real ? fbase + g1.y : -__builtin_inff();
            reinterpret_cast<float*>(shared.chunk[wave][3])[lane] =
                real ? g1.z : (COMPOSITE ? 0.0f : __builtin_inff());
            uint64_t discs = 0;
            if constexpr (COMPOSITE) {
                discs = __ballot(real && g1.z < 0.0f);
                float ahead = before[0];
#pragma unroll
                for (uint32_t q = 1; q < WAVES; ++q) ahead = from == q ? before[q] : ahead;
                reinterpret_cast<float*>(shared.chunkReach[wave])[lane] = fmaxS(ahead, shared.reach[buf][record]);
            }
            waveSync();
            const uint32_t chunkEnd = total - chunk < kLanes ? total - chunk : kLanes;
            for (uint32_t at16 = 0; at16 < chunkEnd; at16 += 16u) {
                float sixteen[3];
#pragma unroll
                for (uint32_t m = 0; m < 3; ++m) sixteen[m] = shflF(form[m], at16 + (lane & 15u));
                const uint32_t of = shflU(record, at16 + (lane >> 2));
                const float channel = reinterpret_cast<const float*>(&shared.colour[buf][of])[lane & 3u];
                walked += walkSixteen<DEPTH_MODE, COMPOSITE, !COMPOSITE && TRACK>(
                    w, chunkEnd - at16, sixteen, channel, pu, pv, shared.chunk[wave], at16 / 4,
                    &shared.chunkReach[wave][COMPOSITE ? at16 / 4 : 0], stopZ, discs >> at16,
                    static_cast<int32_t>(at16));
                if (__ballot(w.t >= kTMin) == 0) break;
            }
            waveSync();
            // the chunk's places become the records' own
            const auto recordAt = [&](int32_t in) {
                return static_cast<uint32_t>(__shfl(static_cast<int>(record), in < 0 ? 0 : in, 64));
            };
            if constexpr (!COMPOSITE && TRACK) {
                const uint32_t of = recordAt(w.lastIn);
                last = w.lastIn >= 0 ? next + of - tileStart + 1u : last;
                w.lastIn = -1;
            }
            if constexpr (DEPTH_MODE == 1) {
                const uint32_t of = recordAt(w.depthIn);
                depthAt = w.depthIn >= 0 ? shared.colour[buf][of].w : depthAt;
                w.depthIn = -1;
            }
            if constexpr (COMPOSITE) {
                const uint32_t of = recordAt(w.opaqueIn);
                if (w.opaqueIn >= 0) {
                    const float4 o = shared.colour[buf][of];
                    oR = o.x, oG = o.y, oB = o.z, oZ = o.w;
                    opaqueHit = true;
                }
                w.opaqueIn = -1;
            }
            walks = __ballot(w.t >= kTMin) != 0;
            if (!walks) break;
        }
        if constexpr (WAVES == 1) {
            if (!walks) break;
        }
    }
    const float r = w.accum[0], g = w.accum[1], b = w.accum[2], depthSum = w.accum[3];
    const float t = COMPOSITE && w.tStopped >= 0.0f ? w.tStopped : w.t;
    // The walk's records, counted on request (the blend's work is 64 lanes x
    // these steps).
    if (walkSteps != nullptr && lane == 0) atomicAdd(walkSteps, walked);
    if constexpr (MODE == kPartial) {
        partialA[lane] = make_float4(r, g, b, depthSum);
        partialB[lane] = make_float2(t, __uint_as_float(last));
        return;
    } else if constexpr (MODE == kResume) {
        *state = WalkState{r, g, b, t, depthSum, depthAt, last, w.t >= kTMin};
        return;
    }
    if (!inside) return;
    if constexpr (COMPOSITE) {
        finishComposite(f, at0, r, g, b, t, depthSum, depthAt, opaqueHit, make_float4(oR, oG, oB, 1.0f), oZ,
                        underHit, underColour, underZ, colour, depth);
    } else {
        finishPixel(f, px, py, r, g, b, t, depthSum, depthAt, last, colour, depth, lastCount, finalT, accum);
    }
}

// A workgroup a block: four waves a 16x16 one, one wave an 8x8 one. The blocks
// of one 32-pixel tile are workgroups b, b + 8, b + 16, b + 24, which the
// dispatcher deals to one XCD, so their gathers of the tile's records share
// that XCD's L2.
template <uint32_t DEPTH_MODE, uint32_t WAVES, bool COMPOSITE, bool TRACK>
__global__ __launch_bounds__(WAVES* kLanes, kWavesPerSimd) void blendKernel(
    FrameParams f, uint32_t slots, const uint32_t* __restrict__ order, const uint2* __restrict__ ranges,
    const uint32_t* __restrict__ pairSlots, const float4* __restrict__ proj, const float4* __restrict__ underColour,
    const float* __restrict__ underDepth, float4* __restrict__ colour, float* __restrict__ depth,
    uint32_t* __restrict__ lastCount, float* __restrict__ finalT, float4* __restrict__ accum,
    uint32_t* __restrict__ walkSteps, const uint32_t* __restrict__ slotOfPair) {
    const uint32_t tiles = f.tilesX * f.tilesY;
    const uint32_t bits = blockBits(f.tileShift);
    const uint32_t part = (blockIdx.x >> 3) & ((1u << bits) - 1u);
    const uint32_t place = (blockIdx.x >> (3u + bits)) * 8u + (blockIdx.x & 7u);
    if (place >= tiles) return;
    const uint32_t tile = order != nullptr ? order[place] : place;
    if (tile >= tiles) return;   // an order entry that is not a tile: draw nothing
    __shared__ BlendShared<WAVES, COMPOSITE> shared;
    const uint2 rg = ranges[tile];
    blendBlock<DEPTH_MODE, WAVES, COMPOSITE, kFinish, TRACK>(
        shared, f, partOrigin(f, tile, part, WAVES == 1 ? 3u : 4u), rg, rg.x, slots, pairSlots, proj, underColour,
        underDepth, colour, depth, lastCount, finalT, accum, nullptr, nullptr, nullptr, walkSteps, slotOfPair);
}

// Every block of every view of a batch (2^bits blocks a tile). As a grid
// (PERSISTENT false) workgroup b is task b, the blocks of a tile going to
// workgroups b, b + 8, b + 16, ... of one XCD; persistent, each workgroup takes
// tasks from a shared counter until none are left (task t: tile t >> bits,
// block t & (2^bits - 1)), so one that drew a light block takes the next
// instead of leaving its slot idle.
template <uint32_t DEPTH_MODE, uint32_t WAVES, bool PERSISTENT, bool TRACK>
__global__ __launch_bounds__(WAVES* kLanes, kWavesPerSimd) void blendViewsKernel(
    const FrameParams* __restrict__ params, const ViewInfo* __restrict__ views, uint32_t viewCount, uint32_t tiles,
    uint32_t bits, uint32_t tasks, uint32_t slots, const uint2* __restrict__ ranges,
    const uint32_t* __restrict__ pairSlots, const float4* __restrict__ proj, uint32_t* __restrict__ lastCount,
    float* __restrict__ finalT, float4* __restrict__ accum, uint32_t* __restrict__ queue,
    const uint32_t* __restrict__ slotOfPair) {
    __shared__ BlendShared<WAVES, false> shared;
    __shared__ uint32_t sTask;
    while (true) {
        uint32_t task, g, part;
        if constexpr (PERSISTENT) {
            __syncthreads();   // the last task's LDS is done with
            if (threadIdx.x == 0) sTask = atomicAdd(queue, 1u);
            __syncthreads();
            task = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(sTask)));
            if (task >= tasks) return;
            g = task >> bits;
            part = task & ((1u << bits) - 1u);
        } else {
            task = blockIdx.x;
            g = (task >> (3u + bits)) * 8u + (task & 7u);
            part = (task >> 3) & ((1u << bits) - 1u);
        }
        if (g < tiles) {
            const ViewInfo& v = views[viewOfTile(views, viewCount, g)];
            const FrameParams& f = params[v.params];
            const uint2 rg = ranges[g];
            blendBlock<DEPTH_MODE, WAVES, false, kFinish, TRACK>(
                shared, f, partOrigin(f, g - v.tileBase, part, WAVES == 1 ? 3u : 4u), rg, rg.x, slots, pairSlots,
                proj, nullptr, nullptr, reinterpret_cast<float4*>(v.colour), v.depth,
                lastCount != nullptr ? lastCount + v.pixelBase : nullptr,
                finalT != nullptr ? finalT + v.pixelBase : nullptr, accum != nullptr ? accum + v.pixelBase : nullptr,
                nullptr, nullptr, nullptr, nullptr, slotOfPair);
        }
        if constexpr (!PERSISTENT) return;
    }
}

// Heaviest tiles first: tiles bucketed by the bit length of their pair count,
// buckets in descending order, tiles in index order inside a bucket. One
// workgroup of 16 waves, wave w owning the w-th sixteenth of the tiles: each
// wave counts its segment's buckets, the counts' prefix over (bucket
// descending, wave ascending) gives each wave its first place in every bucket,
// and each wave walks its segment again handing out places.
constexpr uint32_t kBuckets = 33;
constexpr uint32_t kOrderWaves = 16;
constexpr uint32_t kOrderCached = 32768;   // tiles whose bucket the first walk leaves in LDS for the second

__device__ __forceinline__ uint32_t bucketOf(uint2 rg) {
    return 32u - static_cast<uint32_t>(__clz(rg.y - rg.x));   // 0 for an empty tile
}

// The segments of a tile of `pairs` pairs: one, unless it holds more than
// segmentPairs (0: never split).
__device__ __forceinline__ uint32_t segmentsOf(uint32_t pairs, uint32_t segmentPairs) {
    return segmentPairs == 0 || pairs <= segmentPairs ? 1u : (pairs + segmentPairs - 1u) / segmentPairs;
}

// Exclusive sums over the workgroup of three counts, and their totals.
__device__ __forceinline__ void blockScan3(uint32_t v[3], uint32_t total[3], uint32_t (*sWave)[kOrderWaves]) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t inc[3] = {v[0], v[1], v[2]};
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc[k]), d, 64));
            inc[k] += lane >= d ? o : 0u;
        }
    }
    if (lane == 63)
        for (int k = 0; k < 3; ++k) sWave[k][wave] = inc[k];
    __syncthreads();
    for (int k = 0; k < 3; ++k) {
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < kOrderWaves; ++w) {
            before += w < wave ? sWave[k][w] : 0u;
            all += sWave[k][w];
        }
        total[k] = all;
        v[k] = before + inc[k] - v[k];
    }
}

__global__ __launch_bounds__(kOrderWaves * 64) void tileOrderKernel(const uint2* __restrict__ ranges, uint32_t tiles,
                                                                    uint32_t* __restrict__ order,
                                                                    uint32_t segmentPairs, uint4* __restrict__ tasks,
                                                                    uint4* __restrict__ combine,
                                                                    uint32_t* __restrict__ planCounts) {
    __shared__ uint32_t sCount[kOrderWaves][kBuckets];
    __shared__ uint32_t sStart[kOrderWaves][kBuckets];
    __shared__ uint8_t sBucket[kOrderCached];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    for (uint32_t k = tid; k < kOrderWaves * kBuckets; k += blockDim.x) (&sCount[0][0])[k] = 0;
    __syncthreads();
    const uint32_t segment = (tiles + kOrderWaves * 64 - 1) / (kOrderWaves * 64) * 64;   // whole chunks of 64
    const uint32_t begin = wave * segment;
    const uint32_t end = begin + segment < tiles ? begin + segment : tiles;
    // Eight loads in flight before the first count: one trip to memory for a
    // wave's tiles of a 1080p frame instead of one a chunk.
    constexpr uint32_t kOrderBatch = 8;
    for (uint32_t t0 = begin + lane; t0 < end; t0 += 64 * kOrderBatch) {
        uint2 rg[kOrderBatch];
#pragma unroll
        for (uint32_t b = 0; b < kOrderBatch; ++b) {
            const uint32_t t = t0 + 64 * b;
            rg[b] = t < end ? ranges[t] : make_uint2(0u, 0u);
        }
#pragma unroll
        for (uint32_t b = 0; b < kOrderBatch; ++b) {
            const uint32_t t = t0 + 64 * b;
            if (t < end) {
                const uint32_t bucket = bucketOf(rg[b]);
                if (t < kOrderCached) sBucket[t] = static_cast<uint8_t>(bucket);
                atomicAdd(&sCount[wave][bucket], 1u);
            }
        }
    }
    __syncthreads();
    // Bucket k's first place: the tiles of every heavier bucket; then wave w's
    // within it: the bucket's tiles in the waves before w.
    // One wave: lane k < kBuckets holds bucket k's per-wave counts, scans them
    // over the waves in registers, and takes its bucket's first place as the
    // tiles of the heavier buckets (lanes above it: a suffix sum over lanes).
    if (wave == 0) {
        uint32_t c[kOrderWaves], sum = 0;
#pragma unroll
        for (uint32_t ww = 0; ww < kOrderWaves; ++ww) {
            c[ww] = lane < kBuckets ? sCount[ww][lane] : 0u;
            sum += c[ww];
        }
        uint32_t suffix = sum;   // lanes lane .. 63 (zero past the buckets)
#pragma unroll
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t o = static_cast<uint32_t>(__shfl_down(static_cast<int>(suffix), d, 64));
            suffix += lane + d < 64 ? o : 0u;
        }
        const uint32_t above = suffix - sum;
        if (lane < kBuckets) {
            uint32_t start = above;
#pragma unroll
            for (uint32_t ww = 0; ww < kOrderWaves; ++ww) {
                sStart[ww][lane] = start;
                start += c[ww];
            }
        }
    }
    __syncthreads();
    // Each lane's rank among the lanes of its bucket (six ballots on the
    // bucket's bits give the lanes that share it); the group's last lane then
    // moves the bucket's next place on. The places live in LDS, read and written
    // through a volatile pointer so that every round sees the last one's.
    volatile uint32_t* next = &sStart[wave][0];
    const uint64_t below = (1ull << lane) - 1ull;
    static_assert(kBuckets < 64, "a bucket (and the no-tile mark kBuckets) fits six bits");
    for (uint32_t base = begin; base < end; base += 64) {
        const uint32_t t = base + lane;
        const bool mine = t < end;
        const uint32_t bucket = !mine ? kBuckets : t < kOrderCached ? sBucket[t] : bucketOf(ranges[t]);
        uint64_t same = ~0ull;
#pragma unroll
        for (uint32_t bit = 0; bit < 6; ++bit) {
            const bool set = ((bucket >> bit) & 1u) != 0u;
            const uint64_t vote = __ballot(set);
            same &= set ? vote : ~vote;
        }
        const uint32_t place = mine ? next[bucket] + static_cast<uint32_t>(__popcll(same & below)) : 0u;
        if (mine) order[place] = t;
        if (mine && (same & ~below & ~(1ull << lane)) == 0) next[bucket] = place + 1u;
    }
    if (tasks == nullptr) return;
    // The split plan: tiles in that order, each cut into segmentsOf() segments
    // of near-equal length. tasks[k] = (tile, segment begin, end, partial slot
    // or kNoSlot); combine[m] = (tile, first slot, segments) for each split
    // tile. Each thread takes a run of places; sums over the runs place them.
    __shared__ uint32_t sWave[3][kOrderWaves];
    __syncthreads();   // the order is written
    const uint32_t chunk = (tiles + blockDim.x - 1u) / blockDim.x;
    const uint32_t p0 = tid * chunk < tiles ? tid * chunk : tiles;
    const uint32_t p1 = p0 + chunk < tiles ? p0 + chunk : tiles;
    uint32_t v[3] = {0u, 0u, 0u};   // tasks, partial slots, split tiles
    for (uint32_t p = p0; p < p1; ++p) {
        const uint2 rg = ranges[order[p]];
        const uint32_t n = segmentsOf(rg.y - rg.x, segmentPairs);
        v[0] += n;
        v[1] += n > 1 ? n : 0u;
        v[2] += n > 1 ? 1u : 0u;
    }
    uint32_t total[3];
    blockScan3(v, total, sWave);
    for (uint32_t p = p0; p < p1; ++p) {
        const uint32_t tile = order[p];
        const uint2 rg = ranges[tile];
        const uint32_t len = rg.y - rg.x;
        const uint32_t n = segmentsOf(len, segmentPairs);
        const uint32_t segLen = (len + n - 1u) / n;
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t begin = rg.x + k * segLen < rg.y ? rg.x + k * segLen : rg.y;
            const uint32_t end = begin + segLen < rg.y ? begin + segLen : rg.y;
            tasks[v[0] + k] = make_uint4(tile, begin, end, n > 1 ? v[1] + k : kNoSlot);
        }
        if (n > 1) {
            combine[v[2]] = make_uint4(tile, v[1], n, 0u);
            v[1] += n;
            v[2] += 1;
        }
        v[0] += n;
    }
    if (tid == 0) {
        planCounts[0] = total[0];
        planCounts[1] = total[2];
    }
}

// The tasks of a split plan: task k's quadrants are blocks b, b + 8, b + 16,
// ... of one XCD. A task of an unsplit tile finishes its pixels; a
// segment leaves its partial walk in its slot.
template <uint32_t DEPTH_MODE>
__global__ __launch_bounds__(kLanes, kWavesPerSimd) void blendTasksKernel(FrameParams f, uint32_t slots, const uint4* __restrict__ tasks,
                                                           const uint32_t* __restrict__ planCounts,
                                                           const uint2* __restrict__ ranges,
                                                           const uint32_t* __restrict__ pairSlots,
                                                           const float4* __restrict__ proj,
                                                           float4* __restrict__ colour, float* __restrict__ depth,
                                                           uint32_t* __restrict__ lastCount,
                                                           float* __restrict__ finalT, float4* __restrict__ partialA,
                                                           float2* __restrict__ partialB) {
    const uint32_t qBits = quadBits(f.tileShift);
    const uint32_t quadrant = (blockIdx.x >> 3) & ((1u << qBits) - 1u);
    const uint32_t task = (blockIdx.x >> (3u + qBits)) * 8u + (blockIdx.x & 7u);
    if (task >= planCounts[0]) return;
    __shared__ BlendShared<1, false> shared;
    const uint4 tk = tasks[task];
    const uint32_t tileStart = ranges[tk.x].x;
    if (tk.w == kNoSlot) {
        blendBlock<DEPTH_MODE, 1, false, kFinish>(shared, f, partOrigin(f, tk.x, quadrant, 3u),
                                                  make_uint2(tk.y, tk.z), tileStart, slots, pairSlots, proj, nullptr,
                                                  nullptr, colour, depth, lastCount, finalT, nullptr);
    } else {
        const uint64_t at = ((static_cast<uint64_t>(tk.w) << qBits) + quadrant) * kLanes;
        blendBlock<DEPTH_MODE, 1, false, kPartial>(shared, f, partOrigin(f, tk.x, quadrant, 3u),
                                                   make_uint2(tk.y, tk.z), tileStart, slots, pairSlots, proj, nullptr,
                                                   nullptr, colour, depth, lastCount, finalT, nullptr, nullptr,
                                                   partialA + at, partialB + at);
    }
}

// A split tile's pixels, its segments' partial walks composited front to back:
// rgb += T rgb_s, depth sum += T depth_s, T *= T_s. A pixel whose walk would
// stop inside a segment (T below 1e-4, or the threshold depth crossed) walks
// that segment again from its true state, so it stops where the one walk
// would; the others take the segment whole.
template <uint32_t DEPTH_MODE>
__global__ __launch_bounds__(kLanes, kWavesPerSimd) void combineKernel(FrameParams f, uint32_t slots, const uint4* __restrict__ combine,
                                                        const uint32_t* __restrict__ planCounts,
                                                        const uint2* __restrict__ ranges,
                                                        const uint32_t* __restrict__ pairSlots,
                                                        const float4* __restrict__ proj, float4* __restrict__ colour,
                                                        float* __restrict__ depth, uint32_t* __restrict__ lastCount,
                                                        float* __restrict__ finalT,
                                                        const float4* __restrict__ partialA,
                                                        const float2* __restrict__ partialB) {
    const uint32_t qBits = quadBits(f.tileShift);
    const uint32_t quadrant = blockIdx.x & ((1u << qBits) - 1u);
    const uint32_t c = blockIdx.x >> qBits;
    if (c >= planCounts[1]) return;
    const uint4 ct = combine[c];
    const uint32_t tile = ct.x, n = ct.z, lane = threadIdx.x;
    const uint2 origin = partOrigin(f, tile, quadrant, 3u);
    const uint32_t x0 = origin.x, y0 = origin.y;
    if (x0 >= f.width || y0 >= f.height) return;
    const uint32_t px = x0 + (lane & 7u), py = y0 + (lane >> 3);
    const bool inside = px < f.width && py < f.height && px < x0 + 8u && py < y0 + 8u;
    const uint2 rg = ranges[tile];
    const uint32_t len = rg.y - rg.x, segLen = (len + n - 1u) / n;
    __shared__ BlendShared<1, false> shared;
    WalkState st{0.0f, 0.0f, 0.0f, 1.0f, 0.0f, -1.0f, 0u, inside};
    for (uint32_t k = 0; k < n; ++k) {
        const uint64_t at = ((static_cast<uint64_t>(ct.y + k) << qBits) + quadrant) * kLanes + lane;
        const float4 pa = partialA[at];
        const float2 pb = partialB[at];
        bool again = false;
        if (st.active) {
            const float tEnd = st.t * pb.x;
            again = tEnd < 1e-4f;
            if constexpr (DEPTH_MODE == 1) again = again || (st.depthAt < 0.0f && 1.0f - tEnd >= f.depthThreshold);
            if (!again) {
                st.r = __builtin_fmaf(st.t, pa.x, st.r);
                st.g = __builtin_fmaf(st.t, pa.y, st.g);
                st.b = __builtin_fmaf(st.t, pa.z, st.b);
                st.depthSum = __builtin_fmaf(st.t, pa.w, st.depthSum);
                st.t = tEnd;
                st.last = __float_as_uint(pb.y) != 0u ? __float_as_uint(pb.y) : st.last;
            }
        }
        if (__ballot(again) != 0) {
            const uint32_t begin = rg.x + k * segLen < rg.y ? rg.x + k * segLen : rg.y;
            const uint32_t end = begin + segLen < rg.y ? begin + segLen : rg.y;
            WalkState w = st;
            w.active = again;
            blendBlock<DEPTH_MODE, 1, false, kResume>(shared, f, origin, make_uint2(begin, end), rg.x, slots,
                                                      pairSlots, proj, nullptr, nullptr, colour, depth, lastCount,
                                                      finalT, nullptr, &w);
            if (again) st = w;
            __syncthreads();   // the walk's list is refilled by the next one
        }
    }
    if (!inside) return;
    finishPixel(f, px, py, st.r, st.g, st.b, st.t, st.depthSum, st.depthAt, st.last, colour, depth, lastCount, finalT,
                nullptr);
}

template <uint32_t DEPTH_MODE, bool COMPOSITE>
void launchBlend(const FrameParams& f, uint32_t slots, const uint32_t* order, const uint2* ranges,
                 const uint32_t* pairSlots, const float4* proj, const float4* underColour, const float* underDepth,
                 float4* colour, float* depth, uint32_t* lastCount, float* finalT, float4* accum,
                 hipStream_t stream, uint32_t* walkSteps = nullptr, const uint32_t* slotOfPair = nullptr) {
    // A workgroup a block, the grid rounded up to whole groups of eight tiles.
    // The last contributor is tracked only where it is kept.
    const uint32_t tiles = f.tilesX * f.tilesY;
    const uint32_t blocks = (tiles + 7u) / 8u * (8u << blockBits(f.tileShift));
    const auto go = [&](auto waves, auto track) {
        constexpr uint32_t W = decltype(waves)::value;
        blendKernel<DEPTH_MODE, W, COMPOSITE, decltype(track)::value><<<blocks, W * kLanes, 0, stream>>>(
            f, slots, order, ranges, pairSlots, proj, underColour, underDepth, colour, depth, lastCount, finalT, accum,
            walkSteps, slotOfPair);
    };
    using One = std::integral_constant<uint32_t, 1>;
    using Four = std::integral_constant<uint32_t, 4>;
    if (!COMPOSITE && lastCount != nullptr) {
        if (f.tileShift == 3) go(One{}, std::bool_constant<!COMPOSITE>{}); else go(Four{}, std::bool_constant<!COMPOSITE>{});
    } else {
        if (f.tileShift == 3) go(One{}, std::false_type{}); else go(Four{}, std::false_type{});
    }
}

template <uint32_t DEPTH_MODE>
void launchBlendViews(bool persistent, uint32_t gridCap, const FrameParams* params, const ViewInfo* views,
                      uint32_t viewCount, uint32_t tiles, uint32_t tileShift, uint32_t slots, const uint2* ranges,
                      const uint32_t* pairSlots, const float4* proj, uint32_t* lastCount, float* finalT, float4* accum,
                      uint32_t* queue, hipStream_t stream, const uint32_t* slotOfPair) {
    const uint32_t bits = blockBits(tileShift);
    const auto go = [&](auto waves, auto track) {
        constexpr uint32_t W = decltype(waves)::value;
        constexpr bool T = decltype(track)::value;
        if (persistent) {
            const uint32_t tasks = tiles << bits;
            const uint32_t cap = gridCap / W > 0 ? gridCap / W : 1u;
            const uint32_t grid = tasks < cap ? tasks : cap;
            fill32(queue, 0u, 1, stream);
            blendViewsKernel<DEPTH_MODE, W, true, T><<<grid, W * kLanes, 0, stream>>>(
                params, views, viewCount, tiles, bits, tasks, slots, ranges, pairSlots, proj, lastCount, finalT,
                accum, queue, slotOfPair);
        } else {
            const uint32_t tasks = (tiles + 7u) / 8u * (8u << bits);
            blendViewsKernel<DEPTH_MODE, W, false, T><<<tasks, W * kLanes, 0, stream>>>(
                params, views, viewCount, tiles, bits, tasks, slots, ranges, pairSlots, proj, lastCount, finalT,
                accum, queue, slotOfPair);
        }
    };
    using One = std::integral_constant<uint32_t, 1>;
    using Four = std::integral_constant<uint32_t, 4>;
    if (lastCount != nullptr) {
        if (tileShift == 3) go(One{}, std::true_type{}); else go(Four{}, std::true_type{});
    } else {
        if (tileShift == 3) go(One{}, std::false_type{}); else go(Four{}, std::false_type{});
    }
}

}   // namespace

void blendViews(uint32_t depthMode, bool persistent, uint32_t gridCap, const FrameParams* params,
                const ViewInfo* views, uint32_t viewCount, uint32_t tiles, uint32_t tileShift, uint32_t slots,
                const uint2* ranges,
                const uint32_t* pairSlots, const float4* proj, uint32_t* lastCount, float* finalT, float4* accum,
                uint32_t* queue, hipStream_t stream, const uint32_t* slotOfPair) {
    if (tiles == 0 || viewCount == 0) return;
    if (depthMode == 0) {
        launchBlendViews<0>(persistent, gridCap, params, views, viewCount, tiles, tileShift, slots, ranges, pairSlots,
                            proj, lastCount, finalT, accum, queue, stream, slotOfPair);
    } else {
        launchBlendViews<1>(persistent, gridCap, params, views, viewCount, tiles, tileShift, slots, ranges, pairSlots,
                            proj, lastCount, finalT, accum, queue, stream, slotOfPair);
    }
}

void tileOrder(const uint2* ranges, uint32_t tiles, uint32_t* order, hipStream_t stream) {
    if (tiles == 0) return;
    tileOrderKernel<<<1, kOrderWaves * 64, 0, stream>>>(ranges, tiles, order, 0u, nullptr, nullptr, nullptr);
}

void blendSplit(const FrameParams& f, uint32_t segmentPairs, uint32_t slots, const uint2* ranges,
                const uint32_t* pairSlots, const float4* proj, const BlendPlan& plan, float4* colour, float* depth,
                uint32_t* lastCount, float* finalT, hipStream_t stream) {
    const uint32_t tiles = f.tilesX * f.tilesY;
    if (tiles == 0) return;
    tileOrderKernel<<<1, kOrderWaves * 64, 0, stream>>>(ranges, tiles, plan.order, segmentPairs, plan.tasks,
                                                        plan.combine, plan.counts);
    const uint32_t qBits = quadBits(f.tileShift);
    const uint32_t taskBlocks = (plan.taskCapacity + 7u) / 8u * (8u << qBits);
    const uint32_t combineBlocks = plan.combineCapacity << qBits;
    const auto launch = [&](auto depthMode) {
        constexpr uint32_t D = decltype(depthMode)::value;
        blendTasksKernel<D><<<taskBlocks, kLanes, 0, stream>>>(f, slots, plan.tasks, plan.counts, ranges, pairSlots,
                                                               proj, colour, depth, lastCount, finalT, plan.partialA,
                                                               plan.partialB);
        if (combineBlocks > 0) {
            combineKernel<D><<<combineBlocks, kLanes, 0, stream>>>(f, slots, plan.combine, plan.counts, ranges,
                                                                   pairSlots, proj, colour, depth, lastCount, finalT,
                                                                   plan.partialA, plan.partialB);
        }
    };
    if (f.depthMode == 0) {
        launch(std::integral_constant<uint32_t, 0>{});
    } else {
        launch(std::integral_constant<uint32_t, 1>{});
    }
}

void blend(const FrameParams& f, uint32_t slots, const uint32_t* order, const uint2* ranges,
           const uint32_t* pairSlots, const float4* proj, float4* colour, float* depth, uint32_t* lastCount,
           float* finalT, float4* accum, hipStream_t stream, uint32_t* walkSteps, const uint32_t* slotOfPair) {
    if (f.tilesX * f.tilesY == 0) return;
    if (f.depthMode == 0) {
        launchBlend<0, false>(f, slots, order, ranges, pairSlots, proj, nullptr, nullptr, colour, depth, lastCount,
                              finalT, accum, stream, walkSteps, slotOfPair);
    } else {
        launchBlend<1, false>(f, slots, order, ranges, pairSlots, proj, nullptr, nullptr, colour, depth, lastCount,
                              finalT, accum, stream, walkSteps, slotOfPair);
    }
}

void blendComposite(const FrameParams& f, uint32_t slots, const uint32_t* order, const uint2* ranges,
                    const uint32_t* pairSlots, const float4* proj, const float4* underColour,
                    const float* underDepth, float4* colour, float* depth, hipStream_t stream) {
    if (f.tilesX * f.tilesY == 0) return;
    if (f.depthMode == 0) {
        launchBlend<0, true>(f, slots, order, ranges, pairSlots, proj, underColour, underDepth, colour, depth, nullptr,
                             nullptr, nullptr, stream);
    } else {
        launchBlend<1, true>(f, slots, order, ranges, pairSlots, proj, underColour, underDepth, colour, depth, nullptr,
                             nullptr, nullptr, stream);
    }
}

}   // namespace lrt::kern
