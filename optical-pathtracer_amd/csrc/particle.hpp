// The particle (light-tracing) pass of the renderer: launched by render.hip for the light integrator.
#pragma once

#include <hip/hip_runtime.h>

#include "scene_dev.hpp"

namespace owehip {

struct Settings;

// Exact film splats: each XYZ channel of a pixel is kSplatBins 64-bit integer bins, bin b counting
// units of 2^(kSplatExp0 + 32 b); a float splat adds its 24-bit significand, shifted to its exponent,
// as at most two 32-bit pieces (particle.slang:23-49). Integer sums do not depend on the order
// splats arrive in, so particle images are reproducible bit for bit.
constexpr int kSplatBins = 4;
constexpr int kSplatExp0 = -80;

struct ParticleBatch {
    uint64_t base;              // particle i of the batch is particle base + i of the pass ...
    const uint64_t* index;      // ... or index[i] (device memory) when not null
    uint32_t count, pass;
    unsigned long long* film;   // W·H·3·kSplatBins bins
    double* perParticle;        // when not null: count × 3 XYZ sums per particle instead of the film
    unsigned long long* stats;  // += paths, segments, inconsistencies, leaks
    float invNWY;               // 1 / (NW ∫ȳ)
    // The lane-refill form: particles base + [0, total) of the pass, handed out `chunk` ids at a time
    // from the device counter `next` (zero at launch); a wave starts new particles once `regen` of
    // its lanes are idle.
    uint64_t total;
    unsigned long long* next;
    uint32_t chunk, regen;
};

// Enqueues the batch on `stream`, one thread per particle; stackCap (16, 32 or 48) bounds the BVH
// traversal stack.
void launchParticles(const DScene& sc, const Settings& set, const ParticleBatch& b, uint32_t stackCap,
                     hipStream_t stream);
// Enqueues the pass in the lane-refill form on a grid of `blocks` blocks (the scene's stack bound
// must not exceed 48). sc: the scene's record in device memory. As a kernel argument its hundred
// words are all loaded at the start and spilled to vector lanes, 353 to 425 of them in this kernel: read from memory
// instead, and held to two waves per SIMD where it took the registers of one, the prism's 1,048,576 particles
// with reset and resolve go from 0.80 to 0.70 ms and 16 vcm iterations at 256² from 3.24 to 3.11 ms. (The camera
// paths' persistent kernel is 3 to 5 % faster with the argument.)
void launchParticlesRefill(bool contacts, const DScene* sc, const Settings& set, const ParticleBatch& b, uint32_t blocks,
                           hipStream_t stream);

// How many consecutive ids a lane of the refilling kernels takes when at most `left` are left to a grid of
// `lanes` lanes: `chunk`, but no more than a quarter of a lane's even share. A lane traces its ids one after
// another, so with whole chunks to the end a pass of few ids a lane waits for the lanes that took the last
// ones. `left` is what the asking lane knew at its own last fetch, so it costs no load. Ids stay a partition
// of the pass whatever the grain, and the films are integers, so images do not depend on it. With chunks of 4
// on 768 blocks: pool at 256x192x16 5.3 -> 4.0 ms, a telescope's room at 251x203x16
// 6.0 -> 3.8, light tracing 0.54 -> 0.51. Half a share gives 4.1, 3.9 and 0.51, a whole share 4.6, 5.9 and 0.54;
// chunks of 1 throughout 4.1, 3.8 and 0.51.
__device__ __forceinline__ uint32_t grainOf(uint64_t left, uint32_t chunk, uint32_t lanes) {
    return uint32_t(fmaxf(1.0f, fminf(float(chunk), float(left) / (4.0f * float(lanes)))));
}

}  // namespace owehip
