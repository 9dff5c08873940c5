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
// Enqueues the pass in the lane-refill form on a grid of `blocksPerCU` blocks to each compute unit (the scene's stack
// bound must not exceed 48). scene: sc in device memory. Grids of more than one wave to a SIMD run the kernel held to two,
// which reads the record from memory (the prism's 1,048,576 particles with reset and resolve 0.80 -> 0.70 ms, 16
// vcm iterations at 256² 3.24 -> 3.11; 8,388,608 particles on 4 blocks 3.40 -> 2.30). Smaller grids run the one that
// takes it as an argument and all registers: on 2 and 1 blocks the other one takes 3.66 and 6.67 ms there, this one
// 3.40 and 6.26 (lifted prism 3.28 / 3.22, 5.98 / 5.81). (The camera paths' persistent kernel is 3 to 5 % faster with the
// argument.)
void launchParticlesRefill(const DScene& sc, const DScene* scene, const Settings& set, const ParticleBatch& b,
                           uint32_t computeUnits, uint32_t blocksPerCU, hipStream_t stream);

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
