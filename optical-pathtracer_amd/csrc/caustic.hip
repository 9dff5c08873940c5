// Differentiable caustic design: owe_hip_caustic_* of include/owe_hip_caustic.h.
//
// Forward: one thread per particle, each block over a contiguous range of particles. A particle of
// pass k is stream (hashCombine(seed, i), k): a wavelength importance-sampled over the visible range
// and weighted by the sun's luminous spectrum, and a point on the slab's entry face, stratified over
// square tiles (a wave's particles share a tile or two). It enters at normal incidence (weight 1 − R),
// crosses the slab along +z to the exit surface z = t + h(x, y), refracts out of it (weight 1 − R;
// total internal reflection ends it) and lands on the wall, where its weight spreads over the 3 × 3
// pixels around it with quadratic B-spline weights (continuously differentiable in the landing
// point, so the loss is C¹ in the heights) as 64-bit fixed-point adds — exact, so a pass is
// reproducible.
//
// Backward (path replay): the same particles are drawn again from their seeds and the same float
// operations give the same wall point; the exit's derivatives (by h, h_x and h_y at the particle's exit
// point, exitSlopes) with the spline weights
// and ∂L/∂E at the nine pixels give ∂L/∂(h, h_x, h_y) for this particle. h, h_x and h_y are linear in
// the 4 × 4 heights around the cell (bicubic Hermite patch with central-difference node slopes), so
// the particle adds its share to those sixteen heights: no stored paths. Both passes gather their
// adds (pixels, nodes) in the block's table in LDS and send each touched pixel or node to HBM once
// per block.
//
// Bound by VALU issue and the LDS adds. The patch's weights are products of a row's and a column's
// (16 numbers, not 48), the exit's derivatives follow from the one cosine they depend on, and the
// tile of a particle takes no 64-bit division: 1,048,576 particles, 256² heights, 512² pixels:
// forward 74 → 48 µs, backward 143 → 69 µs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "common.hpp"
#include "owe_hip_caustic.h"
#include "transport_dev.hpp"

using namespace owehip;

namespace owehip {
namespace {

constexpr int kCBlock = 256;
constexpr double kSplatUnits = 4294967296.0;  // fixed-point units per unit of irradiance

struct CArgs {
    const float* heights;
    uint32_t nodes, pixels;
    float slabHalf, z0, zWall, wallHalf;
    float perCell, perPix;   // cells and pixels to a metre
    uint64_t particles, seed, pass;
    DMedium slab, air;
    // The sun's B(λ) / ∫ B ȳ = sunScale e / (λ⁵ (1 − e sunRef)) with e = exp(sunAt − sunC2 / λ), λ in µm: the exponent is
    // taken from that of 555 nm (sunAt; sunRef = exp(−sunAt)), since a cool sun's own leaves float's range.
    float sunScale, sunC2, sunAt, sunRef;
    float tileArea;          // a tile's area / pixel area: with a tile's particle count, irradiance per unit weight
    uint32_t tiles;          // tiles per side (a power of two)
    uint32_t tileShift;      // log2 of all tiles
    double tilesPerParticle;
    unsigned long long* acc;
    float* irradiance;
    const float* gradE;
    float* gradH;
};

// The exit: refraction out of the slab (index n1) into air (n2, η = n1 / n2) through the surface of height
// h and slope (ax, ay) at (x, y), for a ray travelling +z, and the wall point. Snell and Fresnel share their
// cosines c_i = n·(+z) and c_t: r_s = (η c_i − c_t)/(η c_i + c_t), r_p = (c_i − η c_t)/(c_i + η c_t).
// Without contraction, so both passes round it alike.
struct Exit {
    float c, ct, m, idz;  // cos θi, cos θt, the normal's share of the direction, 1 / d_z
    float rs, rp, is, ip;  // the Fresnel amplitudes and their denominators' inverses
    float xw, yw, trans;
};
__device__ __forceinline__ bool exitRay(float h, float ax, float ay, float x, float y, float eta, float z0, float zWall,
                                        Exit& e) {
#pragma clang fp contract(off)
    e.c = invSqrt(ax * ax + ay * ay + 1.0f);
    const float k = 1.0f - eta * eta * (1.0f - e.c * e.c);
    if (!(k >= 0.0f)) return false;  // total internal reflection
    e.ct = sqrtf(k);
    e.m = eta * e.c - e.ct;
    e.idz = quick(1.0f, eta - e.m * e.c);
    const float ds = eta * e.c + e.ct, dp = e.c + eta * e.ct, inv = quick(1.0f, ds * dp);
    e.is = dp * inv;
    e.ip = ds * inv;
    e.rs = e.m * e.is;
    e.rp = (e.c - eta * e.ct) * e.ip;
    e.trans = 1.0f - (e.rs * e.rs + e.rp * e.rp) * 0.5f;
    const float reach = e.m * e.c * e.idz * (zWall - (z0 + h));  // the direction is (m c (ax, ay), d_z)
    e.xw = x + ax * reach;
    e.yw = y + ay * reach;
    return true;
}

// ∂(xw, yw, trans)/∂(h, h_x, h_y) at an exit. The wall point is (x, y) + s(c) (h_x, h_y) L with
// s = m c / d_z, and s and the transmittance depend on the slope through c = (1 + h_x² + h_y²)^(−½) alone:
// ∂c/∂h_x = −h_x c³, c_t' = η² c / c_t, m' = η − c_t', s' = η (m' c + m) / d_z², and each Fresnel amplitude
// (u − v)/(u + v) has the derivative 2 (u' v − u v') / (u + v)².
__device__ __forceinline__ void exitSlopes(const Exit& e, float h, float ax, float ay, float eta, float z0, float zWall,
                                           float dxw[3], float dyw[3], float dT[3]) {
    const float c = e.c, c3 = c * c * c, L = zWall - (z0 + h);
    const float ctp = e.ct > 1e-15f ? quick(eta * eta * c, e.ct) : 0.0f;
    const float s = e.m * c * e.idz, sL = s * L;
    const float q = eta * ((eta - ctp) * c + e.m) * e.idz * e.idz * L * c3;  // −s' L ∂c/∂h_x / h_x
    dxw[0] = -ax * s;
    dxw[1] = sL - q * ax * ax;
    dxw[2] = -q * ax * ay;
    dyw[0] = -ay * s;
    dyw[1] = dxw[2];
    dyw[2] = sL - q * ay * ay;
    const float dTc = 2.0f * eta * (e.ct - c * ctp) * (e.rs * e.is * e.is + e.rp * e.ip * e.ip) * c3;
    dT[0] = 0.0f;
    dT[1] = dTc * ax;
    dT[2] = dTc * ay;
}

// Hermite bases (surfaces.hpp:190-197) at u for the two ends: P, Q and their derivatives.
__device__ __forceinline__ void hermite(float u, float P[2], float Q[2], float dP[2], float dQ[2]) {
    const float u2 = u * u, u3 = u2 * u;
    P[0] = 2.0f * u3 - 3.0f * u2 + 1.0f;
    P[1] = -2.0f * u3 + 3.0f * u2;
    Q[0] = u3 - 2.0f * u2 + u;
    Q[1] = u3 - u2;
    dP[0] = 6.0f * u2 - 6.0f * u;
    dP[1] = -6.0f * u2 + 6.0f * u;
    dQ[0] = 3.0f * u2 - 4.0f * u + 1.0f;
    dQ[1] = 3.0f * u2 - 2.0f * u;
}

// The patch of the cell holding (x, y): the 4 × 4 node block around it, and the weights of its columns
// (x) and rows (y). With central-difference node slopes the Hermite patch is a product: h depends on node
// (r, c) with weight wy[r] wx[c], ∂h/∂u with wy[r] dx[c] and ∂h/∂v with dy[r] wx[c] (u, v in cells).
// Block nodes beyond the grid are its edge's (the edge nodes' one-sided slopes).
struct Patch {
    uint32_t row[4], col[4];  // first node of each row; each column
    float wx[4], dx[4], wy[4], dy[4];
};
__device__ __forceinline__ void patchSide(float f, uint32_t nodes, uint32_t stride, uint32_t at[4], float w[4], float d[4]) {
    const int i = min(max(int(f), 0), int(nodes) - 2);
    float P[2], Q[2], dP[2], dQ[2];
    hermite(f - float(i), P, Q, dP, dQ);
    w[0] = -0.5f * Q[0];
    w[1] = P[0] - 0.5f * Q[1];
    w[2] = P[1] + 0.5f * Q[0];
    w[3] = 0.5f * Q[1];
    d[0] = -0.5f * dQ[0];
    d[1] = dP[0] - 0.5f * dQ[1];
    d[2] = dP[1] + 0.5f * dQ[0];
    d[3] = 0.5f * dQ[1];
#pragma unroll
    for (int k = 0; k < 4; ++k) at[k] = uint32_t(min(max(i - 1 + k, 0), int(nodes) - 1)) * stride;
}
__device__ __forceinline__ void patchAt(const CArgs& a, float x, float y, Patch& p) {
    patchSide((x + a.slabHalf) * a.perCell, a.nodes, 1, p.col, p.wx, p.dx);
    patchSide((y + a.slabHalf) * a.perCell, a.nodes, a.nodes, p.row, p.wy, p.dy);
}

struct Particle {
    float x, y, weight, eta;  // weight: luminous weight × entry transmittance × area factor
};
// The entry face is cut into tiles × tiles square tiles in Morton order; tile t holds the particles
// [⌊t·N/T⌋, ⌊(t+1)·N/T⌋) (T tiles, N particles), each uniform over its tile. Stratified sampling
// (unbiased: each tile's weight is its area over its own count) that also keeps a wave's
// consecutive particles in one small patch of the slab, so their splats and gradient adds meet the
// same pixels and nodes.
__device__ __forceinline__ uint64_t tileStart(uint64_t t, const CArgs& a) { return (t * a.particles) >> a.tileShift; }
__device__ __forceinline__ uint32_t mortonHalf(uint32_t v) {  // the even bits of v, packed
    v &= 0x55555555u;
    v = (v | (v >> 1)) & 0x33333333u;
    v = (v | (v >> 2)) & 0x0F0F0F0Fu;
    v = (v | (v >> 4)) & 0x00FF00FFu;
    v = (v | (v >> 8)) & 0x0000FFFFu;
    return v;
}
__device__ __forceinline__ Particle drawParticle(const CArgs& a, uint64_t i) {
    Rng rng;
    rng.seed(hashPair(a.seed, i), a.pass);
    const float ul = rng.uniform();
    // The visible range's λ (sampleVisibleF) and density: with λ = 538 − atanh(g) / 0.0072 the density's
    // 1 / cosh² is 1 − g².
    const float g = clampf(0.85691062f - 1.82750197f * ul, -0.9705913f, 0.85691062f);
    const float lambda = clampf(538.0f - 138.888889f * atanhf(g), 360.0f, 830.0f);
    const float pdf = 0.0039398042f * (1.0f - g) * (1.0f + g);
    const float u2 = rng.uniform(), u1 = rng.uniform();
    // The tile ⌊i T / N⌋, off by one at most in double, and put right in integers.
    const uint64_t T = uint64_t(1) << a.tileShift;
    uint64_t t = uint64_t(double(i) * a.tilesPerParticle);
    if (t >= T) t = T - 1;
    while (t + 1 < T && tileStart(t + 1, a) <= i) ++t;
    while (t > 0 && tileStart(t, a) > i) --t;
    const uint64_t count = tileStart(t + 1, a) - tileStart(t, a);
    const float side = 2.0f * a.slabHalf / float(a.tiles);
    Particle q;
    q.x = -a.slabHalf + (float(mortonHalf(uint32_t(t))) + u1) * side;
    q.y = -a.slabHalf + (float(mortonHalf(uint32_t(t >> 1))) + u2) * side;
    q.eta = quick(mediumIndex(a.slab, lambda), mediumIndex(a.air, lambda));
    const float r = quick(q.eta - 1.0f, q.eta + 1.0f);  // the entry's Fresnel amplitude at normal incidence
    // B(λ) ȳ(λ) / pdf over the sun's ∫ B ȳ, one quotient of normal numbers for any sun above 100 K (|e's exponent| < 86
    // toward the red; toward the blue e may vanish): Planck's law and cieXYZ's ȳ.
    const float l = lambda * 1e-3f, l2 = l * l;
    auto lobe = [&](float mu, float below, float above) {
        const float u = (lambda - mu) * (lambda < mu ? below : above);
        return expf(-0.5f * u * u);
    };
    const float y = 0.821f * lobe(568.8f, 1.0f / 46.9f, 1.0f / 40.5f) + 0.286f * lobe(530.9f, 1.0f / 16.3f, 1.0f / 31.1f);
    const float e = expf(a.sunAt - quick(a.sunC2, l));
    q.weight = quick(a.sunScale * a.tileArea * y * (1.0f - r * r) * e, l2 * l2 * l * (1.0f - e * a.sunRef) * pdf * float(count));
    return q;
}

// An add to LDS in the block's scope: with atomicAdd the compiler folds it and the add to HBM of a
// crowded table into one through a generic pointer, which is several times slower.
__device__ __forceinline__ void ldsAdd(unsigned long long* p, unsigned long long v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A block's table in LDS of 64-bit integer adds keyed by pixel or node: open addressing over kTableSlots
// (key, sum) pairs. A claimed slot keeps its key, so an add first reads (one read for all lanes of
// a key) and only a first visitor swaps; add is false where kTableProbes slots hold other keys.
// clear and the walk over the claimed slots (take, which empties them) are the whole block's, with a
// barrier between them and any add. Integers, because an LDS float add of a wave takes 200 cycles
// here, with and without lanes on one address, and a 64-bit integer add 28.
constexpr int kTableSlots = 1024;
constexpr int kTableProbes = 8;
constexpr uint32_t kTableEmpty = 0xFFFFFFFFu;

struct BlockTable {
    uint32_t* keys;
    unsigned long long* sums;
    __device__ __forceinline__ void clear() const {
        for (uint32_t q = threadIdx.x; q < uint32_t(kTableSlots); q += kCBlock) {
            keys[q] = kTableEmpty;
            sums[q] = 0;
        }
    }
    __device__ __forceinline__ bool add(uint32_t key, unsigned long long v) const {
        static_assert(kTableSlots == 1 << 10, "the slot hash takes 10 bits");
        uint32_t slot = (key * 2654435761u) >> (32 - 10);
#pragma unroll 1
        for (int probe = 0; probe < kTableProbes; ++probe) {
            uint32_t held = keys[slot];
            if (held == kTableEmpty) held = atomicCAS(&keys[slot], kTableEmpty, key);
            if (held == kTableEmpty || held == key) {
                ldsAdd(&sums[slot], v);
                return true;
            }
            slot = (slot + 1) & uint32_t(kTableSlots - 1);
        }
        return false;
    }
    template <class F>
    __device__ __forceinline__ void take(F&& each) const {
        for (uint32_t q = threadIdx.x; q < uint32_t(kTableSlots); q += kCBlock) {
            const uint32_t key = keys[q];
            if (key == kTableEmpty) continue;
            each(key, sums[q]);
            keys[q] = kTableEmpty;
            sums[q] = 0;
        }
    }
};

// The contiguous range of particles a block takes: ⌈N / blocks⌉ rounded up to whole rounds of its threads.
__device__ __forceinline__ void blockRange(uint64_t n, uint64_t& begin, uint64_t& end) {
    const uint64_t per = ((n + gridDim.x - 1) / gridDim.x + kCBlock - 1) / kCBlock * kCBlock;
    begin = blockIdx.x * per;
    end = begin + per < n ? begin + per : n;
}

__device__ __forceinline__ void heightsAt(const CArgs& a, const Patch& p, float& h, float& fu, float& fv) {
    h = fu = fv = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float hx = 0.0f, dx = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float H = a.heights[p.row[r] + p.col[c]];
            hx += p.wx[c] * H;
            dx += p.dx[c] * H;
        }
        h += p.wy[r] * hx;
        fu += p.wy[r] * dx;
        fv += p.dy[r] * hx;
    }
}

// The splat: a quadratic B-spline over the 3 × 3 pixels about the nearest pixel centre (C¹ in the
// wall point, so the irradiance — and any smooth loss of it — has continuous derivatives): the
// centre pixel (i, j), the offsets t ∈ [−½, ½) from it, and the weights and their derivatives.
__device__ __forceinline__ void splatOf(const CArgs& a, float xw, float yw, int& i, int& j, float wu[3], float wv[3],
                                        float du[3], float dv[3]) {
    const float gu = (xw + a.wallHalf) * a.perPix - 0.5f, gv = (yw + a.wallHalf) * a.perPix - 0.5f;
    const float fi = floorf(gu + 0.5f), fj = floorf(gv + 0.5f);
    i = int(fmaxf(fminf(fi, 1e8f), -1e8f));
    j = int(fmaxf(fminf(fj, 1e8f), -1e8f));
    const float tu = gu - fi, tv = gv - fj;
    wu[0] = 0.5f * (0.5f - tu) * (0.5f - tu);
    wu[1] = 0.75f - tu * tu;
    wu[2] = 0.5f * (0.5f + tu) * (0.5f + tu);
    wv[0] = 0.5f * (0.5f - tv) * (0.5f - tv);
    wv[1] = 0.75f - tv * tv;
    wv[2] = 0.5f * (0.5f + tv) * (0.5f + tv);
    du[0] = -(0.5f - tu);
    du[1] = -2.0f * tu;
    du[2] = 0.5f + tu;
    dv[0] = -(0.5f - tv);
    dv[1] = -2.0f * tv;
    dv[2] = 0.5f + tv;
}

__global__ __launch_bounds__(kCBlock) void causticForward(CArgs a) {
    __shared__ uint32_t keys[kTableSlots];
    __shared__ unsigned long long sums[kTableSlots];
    const BlockTable table{keys, sums};
    table.clear();
    __syncthreads();
    uint64_t begin, end;
    blockRange(a.particles, begin, end);
    for (uint64_t i = begin + threadIdx.x; i < end; i += kCBlock) {
        const Particle q = drawParticle(a, i);
        Patch p;
        patchAt(a, q.x, q.y, p);
        float h, fu, fv;
        heightsAt(a, p, h, fu, fv);
        Exit e;
        if (!exitRay(h, fu * a.perCell, fv * a.perCell, q.x, q.y, q.eta, a.z0, a.zWall, e)) continue;
        const float w = q.weight * e.trans;
        int ci, cj;
        float wu[3], wv[3], du[3], dv[3];
        splatOf(a, e.xw, e.yw, ci, cj, wu, wv, du, dv);
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int pi = ci + c - 1, pj = cj + b - 1;
                if (pi < 0 || pj < 0 || pi >= int(a.pixels) || pj >= int(a.pixels)) continue;
                // Scaling by 2³² is exact in float, so rounding there is rounding the exact product. At the critical
                // angle the transmittance can round below 0: a negative product adds nothing.
                const float scaled = rintf(w * wu[c] * wv[b] * float(kSplatUnits));
                if (!(scaled > 0.0f)) continue;
                const unsigned long long units = (unsigned long long)scaled;
                const uint32_t key = uint32_t(pj) * a.pixels + uint32_t(pi);
                if (!table.add(key, units)) atomicAdd(a.acc + key, units);
            }
    }
    __syncthreads();
    table.take([&](uint32_t key, unsigned long long sum) { atomicAdd(a.acc + key, sum); });
}

__global__ void causticClear(unsigned long long* acc, size_t n) {
    for (size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n; k += size_t(gridDim.x) * blockDim.x) acc[k] = 0;
}
__global__ void causticResolve(const unsigned long long* acc, float* out, size_t n) {
    for (size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n; k += size_t(gridDim.x) * blockDim.x)
        out[k] = float(double(acc[k]) / kSplatUnits);
}
__global__ void causticZero(float* g, size_t n) {
    for (size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n; k += size_t(gridDim.x) * blockDim.x) g[k] = 0.0f;
}

// The gradient adds go through the table as integers in a unit that the block chooses: a round (one
// particle per thread) finds a bound of its adds, and the unit is 2^−kUnitBits of the power of two above
// it (the base). A round more than 2³ above the base or 2⁸ below it empties the table first and chooses
// anew, and so does every kUnitParticles particles, which keeps a sum below 2⁶². An add of fewer
// than float's 24 bits goes to HBM as it is, and so does every add of a round with an infinite
// or undefined one or whose bound no unit suits.
constexpr int kUnitBits = 48;
constexpr uint32_t kUnitParticles = 2048;
__device__ __forceinline__ float blockMax(float v, float* part) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    __syncthreads();  // the previous round's reads of part, and its adds, are done
    if (__lane_id() == 0) part[threadIdx.x / 64] = v;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kCBlock / 64; ++w) v = fmaxf(v, part[w]);
    return v;
}

__global__ __launch_bounds__(kCBlock) void causticBackward(CArgs a) {
    __shared__ uint32_t keys[kTableSlots];
    __shared__ unsigned long long sums[kTableSlots];
    __shared__ float part[kCBlock / 64];
    const BlockTable table{keys, sums};
    table.clear();
    uint64_t begin, end;
    blockRange(a.particles, begin, end);
    constexpr double kMagic = 6755399441055744.0;  // 1.5 · 2⁵²: adding it leaves a rounded integer in the low bits
    float base = 0.0f;                             // the power of two the unit was chosen for; 0: none yet
    double toUnits = 0.0, unit = 0.0;
    uint32_t held = 0;                             // particles the table may hold adds of
    auto flush = [&] {
        table.take([&](uint32_t key, unsigned long long sum) {
            atomicAdd(a.gradH + key, float(double((long long)sum) * unit));
        });
    };
    for (uint64_t first = begin; first < end; first += kCBlock) {  // uniform: whole rounds
        const uint64_t i = first + threadIdx.x;
        Patch p;
        float gh[4] = {}, gu[4] = {}, most = 0.0f;
        const bool live = i < end;
        Exit e;
        float h, fu, fv;
        Particle q;
        bool out = false;
        if (live) {
            q = drawParticle(a, i);
            patchAt(a, q.x, q.y, p);
            heightsAt(a, p, h, fu, fv);
            out = exitRay(h, fu * a.perCell, fv * a.perCell, q.x, q.y, q.eta, a.z0, a.zWall, e);
        }
        if (out) {
            const float ax = fu * a.perCell, ay = fv * a.perCell;
            const float w = q.weight * e.trans;
            int ci, cj;
            float wu[3], wv[3], du[3], dv[3];
            splatOf(a, e.xw, e.yw, ci, cj, wu, wv, du, dv);
            // ∂L/∂(xw, yw, w) from the nine pixels' ∂L/∂E and the spline weights.
            float gx = 0.0f, gy = 0.0f, gw = 0.0f;
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int pi = ci + c - 1, pj = cj + b - 1;
                    if (pi < 0 || pj < 0 || pi >= int(a.pixels) || pj >= int(a.pixels)) continue;
                    const float g = a.gradE[size_t(pj) * a.pixels + pi];
                    gw += g * wu[c] * wv[b];
                    gx += g * du[c] * wv[b];
                    gy += g * wu[c] * dv[b];
                }
            gx *= w * a.perPix;
            gy *= w * a.perPix;
            // ∂L/∂(h, h_x, h_y); the weight depends on them through the exit transmittance.
            float dxw[3], dyw[3], dT[3], gq[3];
            exitSlopes(e, h, ax, ay, q.eta, a.z0, a.zWall, dxw, dyw, dT);
#pragma unroll
            for (int k = 0; k < 3; ++k) gq[k] = gx * dxw[k] + gy * dyw[k] + gw * q.weight * dT[k];
            const float su = gq[1] * a.perCell, sv = gq[2] * a.perCell;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gh[r] = gq[0] * p.wy[r] + sv * p.dy[r];
                gu[r] = su * p.wy[r];
                most = fmaxf(most, fabsf(gh[r]) + 2.0f * fabsf(gu[r]));  // |wx| ≤ 1, |dx| ≤ 2
                if (!(most < __builtin_inff()) || gh[r] != gh[r] || gu[r] != gu[r]) most = __builtin_inff();
            }
        }
        const float top = blockMax(most, part);
        const bool plain = !(top < 1e30f) || top < 1e-30f;
        const bool refit = !plain && (base == 0.0f || top > 8.0f * base || top < 0x1p-8f * base);
        if (refit || held == kUnitParticles) {
            if (base != 0.0f) {
                flush();
                __syncthreads();
            }
            held = 0;
        }
        if (refit) {
            const int ex = int(__float_as_uint(top) >> 23) - 126;  // top < 2^ex
            base = ldexpf(1.0f, ex);
            toUnits = ldexp(1.0, kUnitBits - ex);
            unit = ldexp(1.0, ex - kUnitBits);
        }
        held += kCBlock;
        if (!out) continue;  // no barrier until the next round's
        const float least = base * 0x1p-24f;  // 24 bits
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float g = gh[r] * p.wx[c] + gu[r] * p.dx[c];
                const uint32_t key = p.row[r] + p.col[c];
                if (!plain && fabsf(g) >= least) {
                    const unsigned long long u = (unsigned long long)(__double_as_longlong(fma(double(g), toUnits, kMagic)) -
                                                                      __double_as_longlong(kMagic));
                    if (table.add(key, u)) continue;
                }
                if (g != 0.0f) atomicAdd(a.gradH + key, g);
            }
    }
    __syncthreads();
    if (base != 0.0f) flush();
}

double planck(double lnm, double kelvin) {
    const double c1 = 1.191042972e8, c2 = 1.438776877e4, l = lnm * 1e-3, l2 = l * l;
    return 1e6 * c1 / (l2 * l2 * l * (std::exp(c2 / (l * kelvin)) - 1));
}
double cieYHost(double l) {
    auto lobe = [](double x, double mu, double s1, double s2) {
        const double t = (x - mu) / (x < mu ? s1 : s2);
        return std::exp(-0.5 * t * t);
    };
    return 0.821 * lobe(l, 568.8, 46.9, 40.5) + 0.286 * lobe(l, 530.9, 16.3, 31.1);
}

DMedium toDevMedium(const owe_medium& m) {
    DMedium d{};
    d.indexKind = m.index_kind;
    d.terms = m.terms;
    d.relAir = m.rel_air;
    for (int k = 0; k < 4; ++k) {
        d.a[k] = float(m.coeff_a[k]);
        d.b[k] = float(m.coeff_b[k]);
    }
    return d;
}

// Tiles per side of the entry face: the largest power of two up to 64 that leaves at least 64
// particles per tile.
uint32_t causticTiles(uint64_t particles) {
    uint32_t g = 1;
    while (g < 64 && uint64_t(4) * g * g * 64 <= particles) g *= 2;
    return g;
}

void checkSettings(const owe_caustic_settings& s) {
    require(s.nodes >= 4 && s.nodes <= 8192, "nodes per side must lie in [4, 8192]");
    require(s.pixels >= 2 && s.pixels <= 8192, "pixels per side must lie in [2, 8192]");
    require(s.particles >= 1 && s.particles <= (uint64_t(1) << 34), "particles must lie in [1, 2^34]");
    require(s.slab_half > 0 && s.thickness > 0 && s.wall_half > 0, "sizes must be positive");
    require(s.wall_z > s.thickness, "the wall must lie beyond the slab");
    require(s.sun_kelvin > 100, "sun temperature must exceed 100 K");
    require(s.medium.index_kind >= OWE_INDEX_CONSTANT && s.medium.index_kind <= OWE_INDEX_CIDDOR, "unknown index model");
}

// The kernels' arguments for settings s (everything but the per-call buffers and pass).
CArgs makeArgs(const owe_caustic_settings& s) {
    CArgs a{};
    a.nodes = s.nodes;
    a.pixels = s.pixels;
    a.slabHalf = float(s.slab_half);
    a.z0 = float(s.thickness);
    a.zWall = float(s.wall_z);
    a.wallHalf = float(s.wall_half);
    a.perCell = float((s.nodes - 1) / (2 * s.slab_half));
    a.perPix = float(s.pixels / (2 * s.wall_half));
    a.particles = s.particles;
    a.seed = s.seed;
    a.slab = toDevMedium(s.medium);
    owe_medium air{};
    air.index_kind = OWE_INDEX_CIDDOR;
    a.air = toDevMedium(air);
    // ∫ B ȳ dλ over 360–830 nm (composite Simpson, 0.5 nm).
    const int n = 940;
    const double hh = 470.0 / n;
    double sum = planck(360.0, s.sun_kelvin) * cieYHost(360.0) + planck(830.0, s.sun_kelvin) * cieYHost(830.0);
    for (int k = 1; k < n; ++k) {
        const double l = 360.0 + k * hh;
        sum += planck(l, s.sun_kelvin) * cieYHost(l) * ((k & 1) ? 4 : 2);
    }
    a.sunC2 = float(1.438776877e4 / s.sun_kelvin);
    a.sunAt = float(1.438776877e4 / (0.555 * s.sun_kelvin));
    a.sunRef = float(std::exp(-double(a.sunAt)));
    a.sunScale = float(1e6 * 1.191042972e8 * std::exp(-double(a.sunAt)) / (sum * hh / 3));
    const double pix = 2 * s.wall_half / s.pixels;
    a.tiles = causticTiles(s.particles);
    while ((uint64_t(1) << a.tileShift) < uint64_t(a.tiles) * a.tiles) ++a.tileShift;
    a.tilesPerParticle = double(uint64_t(1) << a.tileShift) / double(s.particles);
    const double side = 2 * s.slab_half / a.tiles;
    a.tileArea = float(side * side / (pix * pix));
    return a;
}

// The most blocks of 256 a pass runs on: 8 per compute unit.
int passGrid(int device) {
    int cus = 0;
    OWE_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    require(cus > 0, "cannot read the device's compute-unit count");
    return cus * 8;
}
// The blocks of a pass of n particles: no more than give each thread one.
dim3 passBlocks(int most, uint64_t n) {
    return dim3{unsigned(std::min<uint64_t>(uint64_t(most), (n + kCBlock - 1) / kCBlock))};
}

}  // namespace
}  // namespace owehip

struct owe_hip_caustic {
    int device = 0;
    owe_caustic_settings settings{};
    CArgs args{};
    unsigned long long* acc = nullptr;
    int grid = 1024;
};

extern "C" {

int owe_hip_caustic_create(int device, const owe_caustic_settings* settings, owe_hip_caustic** out) {
    owe_hip_caustic* c = nullptr;
    const int st = guard([&] {
        require(settings != nullptr && out != nullptr, "null argument");
        *out = nullptr;
        const owe_caustic_settings& s = *settings;
        checkSettings(s);
        selectDevice(device);
        c = new owe_hip_caustic;
        c->device = device;
        c->settings = s;
        c->grid = passGrid(device);
        c->args = makeArgs(s);
        void* p = nullptr;
        OWE_HIP_CHECK(hipMalloc(&p, size_t(s.pixels) * s.pixels * sizeof(unsigned long long)));
        c->acc = static_cast<unsigned long long*>(p);
        c->args.acc = c->acc;
        *out = c;
    });
    if (st != OWE_HIP_OK && c) {
        if (c->acc) (void)hipFree(c->acc);
        delete c;
    }
    return st;
}

int owe_hip_caustic_destroy(owe_hip_caustic* c) {
    return guard([&] {
        if (!c) return;
        (void)hipSetDevice(c->device);
        OWE_HIP_CHECK(hipDeviceSynchronize());
        if (c->acc) OWE_HIP_CHECK(hipFree(c->acc));
        delete c;
    });
}

int owe_hip_caustic_forward(owe_hip_caustic* c, const float* heights, float* irradiance, uint64_t pass, void* stream) {
    return guard([&] {
        require(c != nullptr && heights != nullptr && irradiance != nullptr, "null argument");
        requireDevicePointer(heights, "heights");
        requireDevicePointer(irradiance, "irradiance");
        OWE_HIP_CHECK(hipSetDevice(c->device));
        const hipStream_t s = static_cast<hipStream_t>(stream);
        CArgs a = c->args;
        a.heights = heights;
        a.pass = pass;
        a.irradiance = irradiance;
        const size_t n = size_t(a.pixels) * a.pixels;
        hipLaunchKernelGGL(causticClear, dim3{1024}, dim3{256}, 0, s, c->acc, n);
        hipLaunchKernelGGL(causticForward, passBlocks(c->grid, a.particles), dim3{kCBlock}, 0, s, a);
        hipLaunchKernelGGL(causticResolve, dim3{1024}, dim3{256}, 0, s, c->acc, irradiance, n);
        OWE_HIP_CHECK(hipGetLastError());
    });
}

int owe_hip_caustic_backward(owe_hip_caustic* c, const float* heights, const float* grad_irradiance, float* grad_heights,
                             uint64_t pass, void* stream) {
    return guard([&] {
        require(c != nullptr && heights != nullptr && grad_irradiance != nullptr && grad_heights != nullptr,
                "null argument");
        requireDevicePointer(heights, "heights");
        requireDevicePointer(grad_irradiance, "grad_irradiance");
        requireDevicePointer(grad_heights, "grad_heights");
        OWE_HIP_CHECK(hipSetDevice(c->device));
        const hipStream_t s = static_cast<hipStream_t>(stream);
        CArgs a = c->args;
        a.heights = heights;
        a.pass = pass;
        a.gradE = grad_irradiance;
        a.gradH = grad_heights;
        hipLaunchKernelGGL(causticZero, dim3{1024}, dim3{256}, 0, s, grad_heights, size_t(a.nodes) * a.nodes);
        hipLaunchKernelGGL(causticBackward, passBlocks(c->grid, a.particles), dim3{kCBlock}, 0, s, a);
        OWE_HIP_CHECK(hipGetLastError());
    });
}

// The allocation-free forward. Its fixed-point bins live in `scratch`, one array per device for the
// life of the process (2 MiB: 512 × 512 pixels at most). Host code never passes the array's name to
// a kernel (in host code it names a host-side stand-in, not device memory): the first call on a
// device, with that device current, asks the runtime for the array's device address and keeps it,
// and every later call on that device uses the kept address. Every call clears the bins it uses
// before splatting; calls that overlap on one device share the array and race.
static __device__ __align__(256) unsigned long long scratch[size_t(OWE_CAUSTIC_NOALLOC_MAX_PIXELS)];

namespace {

constexpr int kMaxDevices = 64;

struct ScratchSlot {
    unsigned long long* bins = nullptr;
    int grid = 0;
};

ScratchSlot scratchFor(int device) {
    static std::mutex mu;
    static ScratchSlot slots[kMaxDevices];
    require(device < kMaxDevices, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(mu);
    ScratchSlot& s = slots[device];
    if (!s.bins) {
        void* p = nullptr;
        OWE_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        require(p != nullptr, "the scratch array has no device address");
        s.grid = passGrid(device);
        s.bins = static_cast<unsigned long long*>(p);
    }
    return s;
}

}  // namespace

int owe_hip_caustic_forward_noalloc(int device, const owe_caustic_settings* settings, const float* heights,
                                    float* irradiance, uint64_t pass, void* stream) {
    return guard([&] {
        require(settings != nullptr && heights != nullptr && irradiance != nullptr, "null argument");
        const owe_caustic_settings& s = *settings;
        checkSettings(s);
        const size_t n = size_t(s.pixels) * s.pixels;
        if (n > size_t(OWE_CAUSTIC_NOALLOC_MAX_PIXELS))
            fail(OWE_HIP_ERR_INVALID, "the allocation-free forward holds at most " +
                                          std::to_string(OWE_CAUSTIC_NOALLOC_MAX_PIXELS) + " pixels (512 x 512); " +
                                          std::to_string(s.pixels) + " x " + std::to_string(s.pixels) + " asked");
        selectDevice(device);
        requireDevicePointer(heights, "heights", device);
        requireDevicePointer(irradiance, "irradiance", device);
        const ScratchSlot slot = scratchFor(device);
        CArgs a = makeArgs(s);
        a.acc = slot.bins;
        a.heights = heights;
        a.pass = pass;
        a.irradiance = irradiance;
        const hipStream_t st = static_cast<hipStream_t>(stream);
        hipLaunchKernelGGL(causticClear, dim3{1024}, dim3{256}, 0, st, slot.bins, n);
        hipLaunchKernelGGL(causticForward, passBlocks(slot.grid, a.particles), dim3{kCBlock}, 0, st, a);
        hipLaunchKernelGGL(causticResolve, dim3{1024}, dim3{256}, 0, st, slot.bins, irradiance, n);
        OWE_HIP_CHECK(hipGetLastError());
    });
}

}  // extern "C"
