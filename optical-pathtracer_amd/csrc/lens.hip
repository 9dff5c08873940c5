// Batched lens analysis: owe_hip_lens_batch_* of include/owe_hip_lens.h.
//
// Work is a flat list of items — (lens, wavelength, block of `raysPerItem` rays) — drained by a
// persistent grid: each block takes the next few items with one atomic, its threads trace an item's rays
// through the lens surface after surface, reduce the spot's sums across each wave in double and add
// them to the (lens, wavelength) totals with one atomic per sum; arrived rays also land on the lens's
// through-focus stack of detector grids as 64-bit fixed-point weights, so the irradiance is
// independent of order. The grid adds gather first in the block's hash table in LDS (bin → sum),
// flushed to HBM when its items move to another lens: most of a lens's rays meet a bin already in
// the table and HBM sees about one atomic per bin touched instead of one per ray. Lenses of very
// different ray counts (4k to 1M) share the launch without tails of idle blocks.
//
// Ray–surface roots follow SagSurface (src/owe/scene/geometry.cpp:115-166,
// src/owe/core/shared/surfaces.hpp:13-94) with the reference's float tolerances. A conic or flat row is met from
// its vertex plane by the small root (conicHit): in float64 on a steep surface (|c|·r_max > 0.5) and
// throughout instruments with mirrors or without focal power (metre paths, high angular magnification), in
// float32 elsewhere. Where another root may come first, and on aspheres, sagHit decides: a float quadric root
// re-solved from the approximate hit point, a numeric asphere root polished by Newton steps in float64. Gaps
// between rows are subtracted in double and the spot sums accumulated in double. Transmission is the walk's
// deterministic refraction with weight T = 1 − R (transport.cpp:531-595); TIR or a missed aperture
// ends a ray.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"
#include "owe_hip_lens.h"
#include "shapes_dev.hpp"
#include "transport_dev.hpp"

using namespace owehip;

namespace owehip {
namespace {

constexpr int kLensBlock = 256;
constexpr int kResidentBlocks = 3;  // blocks to a compute unit that registers and LDS hold
constexpr double kHistScale = 4294967296.0;  // 2^32 units of weight per unit
// A block's bin table: open addressing over kHashSlots (bin, sum) pairs, at most kHashProbes probes
// before an add goes straight to HBM. An aberrated lens's five planes touch 1,000 bins and more: a table
// of 512 slots to each wave was crowded and sent most adds to HBM (the kernel waited on them for
// two thirds of its time), while 48 KiB to a block leave the three blocks to a compute unit that its registers allow.
constexpr int kHashSlots = 4096;
constexpr int kHashProbes = 8;
constexpr uint32_t kPlaneGroup = 8;
constexpr uint32_t kHashEmpty = 0xFFFFFFFFu;
// The steepness |c|·r_max above which a quadric root is polished in float64.
constexpr double kSteepPolish = 0.5;

// A lens row: its sag surface (shapes_dev.hpp; a mirror's annulus outside its hole), the vertex
// position along the fixed chart, and whether it reflects.
struct DSurf : DSag {
    float z;
    float gap;  // signed distance along the chart to the next row's vertex
    double gapD;
    int32_t reflect;
};

// Parameters differentiated per gradient pass (of up to OWE_LENS_MAX_PARAMS), and the sums a pass
// adds per (lens, wavelength, parameter): ΣA', ΣB' (x, y), ΣA·A', ΣB·B', Σ(A'·B + A·B').
constexpr int kGroup = 4;
constexpr int kGradSums = 7;

struct DLensInfo {
    uint32_t first, count;    // surfaces
    uint64_t rays;            // per wavelength
    uint64_t itemBase;        // first work item
    uint32_t itemsPerLambda;
    uint32_t rings;           // 0: Fibonacci lattice; r: hexapolar rings
    double rEP, zEP, zStart;  // entrance pupil (sampling radius 0.999 rEP) and launch plane
    double yStart;            // the launch plane's offset in y of a pupil point's ray
    float detX, detY, detZ, detHalf;  // detector grid centre, plane, half size (0: no grid)
    float detScale;           // pixels per metre of the grid
    float detStep;            // through-focus plane spacing along z
    float refB;               // afocal: a slope near the rays' (the paraxial apparent angle's) and its angle
    double refA;
    int32_t afocal;           // spot sums of angles (afocalSpot) instead of (A, B) at an image
    int32_t mirrors;          // reflecting rows: their vertex planes obstruct
    uint64_t mirrorMask;      // which of the first 64 rows reflect
};

struct LensArgs {
    const DSurf* surf;
    const DLensInfo* lens;
    const float* eta;         // [surface × nλ]: index before over index after each surface
    uint32_t nLenses, nLambda, raysPerItem, pixels, planes;
    uint32_t chunk;           // consecutive items a block takes at a time
    uint64_t totalItems;
    double dirY, dirZ;        // collimated field direction (0, sin θ, cos θ)
    unsigned long long* next;
    double* moments;          // [lens × nλ × OWE_LENS_MOMENTS]
    unsigned long long* hist; // [lens × planes × pixels²]
    // Gradient passes: parameters [paramBase, paramBase + kGroup) of nParams, each (surface within
    // the lens, field); their sums [lens × nλ × OWE_LENS_MAX_PARAMS × kGradSums].
    uint32_t nParams, paramBase;
    int32_t paramSurface[OWE_LENS_MAX_PARAMS], paramField[OWE_LENS_MAX_PARAMS];
    double* grads;
    int32_t sums;             // a gradient pass also adds the moments and histogram
};

// Pupil point i of n on the entrance pupil of radius rEP, in double: a Fibonacci lattice over the
// disc of radius 0.999 rEP, or with rings > 0 spotAt's hexapolar pattern (analysis.cpp:124-131) —
// point 0 the centre, ring k holding the 6k points after the 1 + 3k(k − 1) before it.
__device__ __forceinline__ void pupilPoint(uint64_t i, uint64_t n, uint32_t rings, double rEP, double& x, double& y) {
    if (rings > 0) {
        if (i == 0) {
            x = y = 0.0;
            return;
        }
        uint64_t k = uint64_t((3.0 + sqrt(12.0 * double(i) - 3.0)) / 6.0);
        while (k > 1 && 1 + 3 * k * (k - 1) > i) --k;
        while (1 + 3 * k * (k + 1) <= i) ++k;
        const uint64_t j = i - (1 + 3 * k * (k - 1)), m = 6 * k;
        const double rr = rEP * double(k) / double(rings) * 0.999;
        const double a = 2.0 * 3.14159265358979323846 * double(j) / double(m);
        x = rr * cos(a);
        y = rr * sin(a);
        return;
    }
    // The lattice in float: the golden-ratio fraction of i from 64-bit fixed point (exact for any
    // i), the radius and angle to float rounding.
    const float rr = 0.999f * float(rEP) * quickSqrt(quick(float(i) + 0.5f, float(n)));
    const float f = float(uint32_t((i * 0x9E3779B97F4A7C15ull) >> 40)) * 0x1p-24f;
    float sa, ca;
    sincospif(2.0f * f, &sa, &ca);
    x = double(rr * ca);
    y = double(rr * sa);
}

// Whether the ray from o along d, up to z = zEnd, crosses the vertex-plane annulus hole ≤ r ≤
// semi-diameter of a mirror of the lens other than rows `from` and `to`. Only mirrors' rows are read:
// those of the first 64 rows from the lens's mask, any later ones by looking.
__device__ __forceinline__ bool obstructs(const DSurf& m, f3 o, f3 d, float zEnd) {
    if (!(m.z > fminf(o.z, zEnd) && m.z < fmaxf(o.z, zEnd))) return false;
    const float s = (m.z - o.z) / d.z;
    const float x = o.x + d.x * s, y = o.y + d.y * s, r2 = x * x + y * y;
    return r2 >= m.rMin2 && r2 <= m.rMax2;
}
__device__ __forceinline__ bool obstructed(const LensArgs& a, const DLensInfo& L, f3 o, f3 d, float zEnd, uint32_t from,
                                           uint32_t to) {
    if (d.z == 0.0f) return false;
    for (uint64_t left = L.mirrorMask; left != 0; left &= left - 1) {
        const uint32_t j = uint32_t(__ffsll((long long)left)) - 1;
        if (j != from && j != to && obstructs(a.surf[L.first + j], o, d, zEnd)) return true;
    }
    for (uint32_t j = 64; j < L.count; ++j)
        if (j != from && j != to && a.surf[L.first + j].reflect && obstructs(a.surf[L.first + j], o, d, zEnd)) return true;
    return false;
}

// Derivatives of the ray with respect to the kGroup parameters of a gradient pass.
struct RayGrad {
    float o[3][kGroup], d[3][kGroup];
};

// A conic or flat row met from o (z from its vertex) along unit d: from the vertex plane z = 0, where the
// quadric c (x² + y² + (1 + k) z²) = 2 z has the constant term c (x² + y²) and its root on the vertex's sheet
// is the small one C / w, which loses no digits; T: float, or double on rows with polish64. N is the
// unnormalised normal (−c x, −c y, 1 − (1 + k) c z). The other root w / A is no crossing of this row where
// there is none (A = 0), where it lies on the conic's other sheet, or behind o. kHit: the small root is the
// first crossing; kMiss: the ray does not cross the row; kOther: neither is shown (the ray's z-part does
// not dominate at the vertex plane, or the other root may be a crossing that comes first or alone), and
// sagHit decides.
enum { kMiss, kHit, kOther };
template <class T>
__device__ __forceinline__ int conicHit(const DSurf& sf, T c, T ck, T ox, T oy, T oz, T dx, T dy, T dz, float& th, f3& q,
                                        f3& N) {
    const T tv = -oz / dz;  // correctly rounded: to the first row all rays share it, and an ulp would shift every one in y
    const T x0 = ox + dx * tv, y0 = oy + dy * tv;
    const T A = c * (dx * dx + dy * dy) + ck * dz * dz;
    const T B = c * (x0 * dx + y0 * dy) - dz;
    const T C = c * (x0 * x0 + y0 * y0);
    const T disc = B * B - A * C;
    if (!(B * dz < T(0))) return kOther;
    if (disc < T(0)) return kMiss;
    const T w = -(B + copysign(quickSqrt(disc), B));
    const T t2 = quick(C, w), t = tv + t2;
    const T x = ox + dx * t, y = oy + dy * t, z = dz * t2;  // one rounding each
    q = mk3(float(x), float(y), float(z));
    N = mk3(float(-c * x), float(-c * y), float(T(1) - ck * z));
    th = float(t);
    const bool first = A * dz < T(0);  // the other root comes before this one
    const bool none = A == T(0) || ck * dz * w * A > T(1.001) * A * A || (first && (tv * A + w) * w > T(1e-3) * w * w);
    const bool fits = t > T(0) && sagAccept(sf, q) && N.z >= -1e-6f;
    if (fits) return first && !none ? kOther : kHit;
    return none ? kMiss : kOther;
}

// One ray i of lens L at wavelength w: true when every surface takes it — a refracting row refracts
// it, a mirror reflects it — no mirror body stops it and it leaves along +z; p, d after the last
// surface. With kGrad the derivatives of p and d ride along (launch rays held fixed): at each
// surface the implicit function theorem on F = sag(r²) − z gives the root's derivative
// dt = −(∇F·(do + t dd) + dz_v + F_θ)/F_t, the hit point dp = do + t dd + dt d, the normal's through
// dN of N = (−2g x, −2g y, 1) with g = d sag / d r², and the refracted or reflected direction's by
// the chain rule of its formula. A parameter of a later row has no derivative yet and is skipped
// (uniformly: 37 of 48 row-parameter pairs are left of the Gregorian's eight).
// Bound by VALU issue. The vertex-plane root, one cosine for Fresnel and Snell, one division for both
// Fresnel amplitudes and the second-order renormalisation take about a third of the instructions of
// the general quadric with its second solve (refineRoot) and separate formulas, and lie closer to the
// 64-bit trace: 64 achromats (84 M rays, five planes) 5.87 → 3.14 ms; 32 Gregorians with eight
// derivatives 2.54 → 1.38 ms. Errors against the 64-bit trace, general quadric and correctly rounded formulas
// → these (4.1 M rays of 48 achromats, rms): point 6.20e-10 → 6.10e-10 m, direction 2.7e-8 → 2.2e-8,
// transmittance 3.8e-8 → 3.1e-8, intercept at z = 0 7.79e-10 both; Gregorians' direction 6.2e-7 → 3.9e-7. (An
// estimate for −oz / dz shifted all rays by 2.7e-11 m in y; x0 + dx t2 for x took the point to 6.16e-10.)
template <bool kGrad>
__device__ __forceinline__ bool traceLensRay(const LensArgs& a, const DLensInfo& L, uint32_t w, uint64_t i, f3& p, f3& d,
                                             float& T, RayGrad& G) {
    double px, py;
    pupilPoint(i, L.rays, L.rings, L.rEP, px, py);
    // o: z from the vertex of the row to be met, oz the same in double for rows with polish64 (a gap's
    // rounding to float defocuses a high magnification by 10⁻⁴ of its spot).
    f3 o = mk3(float(px), float(py + L.yStart), float(L.zStart));
    double oz = L.zStart;
    d = mk3(0.0f, float(a.dirY), float(a.dirZ));
    T = 1.0f;
    if (kGrad) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int k = 0; k < kGroup; ++k) G.o[c][k] = G.d[c][k] = 0.0f;
    }
    for (uint32_t k = 0; k < L.count; ++k) {
        const DSurf& sf = a.surf[L.first + k];
        f3 q, n;
        float th;
        int met = kOther;
        if (sf.nA == 0) {
            f3 N;
            met = sf.polish64 ? conicHit<double>(sf, sf.c, sf.ck, o.x, o.y, oz, d.x, d.y, d.z, th, q, N)
                              : conicHit<float>(sf, sf.cf, sf.ckf, o.x, o.y, o.z, d.x, d.y, d.z, th, q, N);
            if (met == kMiss) return false;
            n = N * invSqrt(dot3(N, N));
        }
        if (met == kOther) {
            if (!sagHit(sf, o, d, 0.0f, __builtin_inff(), false, th, q)) return false;
            n = sagNormalF(sf, q);
        }
        if (L.mirrors && obstructed(a, L, mk3(o.x, o.y, o.z + sf.z), d, q.z + sf.z, k == 0 ? L.count : k - 1, k)) return false;
        const float dn = dot3(d, n);
        const float eta = sf.reflect ? 1.0f : a.eta[(L.first + k) * a.nLambda + w];
        float ct = 0.0f;
        f3 wv;
        if (sf.reflect) {
            wv = d - n * (2.0f * dn);
        } else {
            // Snell and Fresnel share the cosines: r_s = (η c_i − c_t)/(η c_i + c_t), r_p = (c_i − η c_t)/(c_i + η c_t).
            const float ci = fminf(fabsf(dn), 1.0f), k2 = 1.0f - eta * eta * (1.0f - ci * ci);
            if (k2 < 0.0f) return false;
            ct = quickSqrt(k2);
            const float ps = eta * ci + ct, pp = ci + eta * ct;
            const float inv = quick(1.0f, ps * pp);
            const float rs = (eta * ci - ct) * pp * inv, rp = (ci - eta * ct) * ps * inv;
            T -= T * fminf(0.5f * (rs * rs + rp * rp), 1.0f);  // at the critical angle the sum can round past 2
            const f3 u = d * eta + n * (copysignf(ct, dn) - eta * dn);
            wv = u * (1.5f - 0.5f * dot3(u, u));  // |u| = 1 to rounding
        }
        if (kGrad) {
            // The surface's partials at the local hit point q.
            const float r2 = q.x * q.x + q.y * q.y, c = sf.cf, kk = sf.kf;
            const float S2 = fmaxf(1e-30f, 1.0f - (1.0f + kk) * c * c * r2), iS = invSqrt(S2), S = S2 * iS;
            const float i1 = quick(1.0f, 1.0f + S), iS3 = iS * iS * iS, c3 = c * c * c;
            float g = 0.5f * c * iS, gr = 0.25f * (1.0f + kk) * c3 * iS3;
            const float Fc = r2 * ((1.0f + S) + (1.0f + kk) * r2 * c * c * iS) * i1 * i1;
            const float Fk = 0.5f * c3 * r2 * r2 * iS * i1 * i1;
            const float gc = 0.5f * (iS + (1.0f + kk) * c * c * r2 * iS3);
            const float gk = 0.25f * c3 * r2 * iS3;
            float FA[4], gA[4], rj = 1.0f;  // rj = r2^j
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                FA[j] = rj * r2 * r2;                   // ∂sag/∂A_j = r2^(2+j)
                gA[j] = float(2 + j) * rj * r2;         // ∂g/∂A_j = (2+j) r2^(1+j)
                if (j < sf.nA) {
                    g += sf.A[j] * gA[j];
                    gr += sf.A[j] * float(2 + j) * float(1 + j) * rj;
                }
                rj *= r2;
            }
            const f3 gradF = mk3(2.0f * g * q.x, 2.0f * g * q.y, -1.0f);
            const float iFt = quick(1.0f, dot3(gradF, d));
            const f3 N = mk3(-2.0f * g * q.x, -2.0f * g * q.y, 1.0f);
            const float invN = invSqrt(dot3(N, N));
            const float sig = dn < 0.0f ? 1.0f : -1.0f;  // the refraction's facing normal
            const float ci = fabsf(dn), kd = ct > 1e-15f ? quick(eta * eta * ci, ct) : 0.0f;  // d c_t = kd · d c_i
#pragma unroll
            for (int kp = 0; kp < kGroup; ++kp) {
                const uint32_t pi = a.paramBase + uint32_t(kp);
                if (pi >= a.nParams || uint32_t(a.paramSurface[pi]) > k) continue;
                const uint32_t ps = uint32_t(a.paramSurface[pi]);
                const int pf = a.paramField[pi];
                const float dzv = pf == OWE_LENS_PARAM_THICKNESS && ps < k ? 1.0f : 0.0f;
                float Fth = 0.0f, gth = 0.0f;
                if (ps == k) {
                    if (pf == OWE_LENS_PARAM_CURVATURE) Fth = Fc, gth = gc;
                    if (pf == OWE_LENS_PARAM_CONIC) Fth = Fk, gth = gk;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (pf == OWE_LENS_PARAM_A4 + j) Fth = FA[j], gth = gA[j];
                }
                const f3 dO = mk3(G.o[0][kp], G.o[1][kp], G.o[2][kp]), dD = mk3(G.d[0][kp], G.d[1][kp], G.d[2][kp]);
                const f3 dx = dO + dD * th;
                const float dt = -(dot3(gradF, dx) + dzv + Fth) * iFt;
                const f3 dP = dx + d * dt;
                // dN from dg = gr dr² + g_θ and the local point's move.
                const float dg = gr * 2.0f * (q.x * dP.x + q.y * dP.y) + gth;
                const f3 dN = mk3(-2.0f * (dg * q.x + g * dP.x), -2.0f * (dg * q.y + g * dP.y), 0.0f);
                const f3 dnv = (dN - n * dot3(n, dN)) * invN;
                f3 dW;
                if (sf.reflect) {
                    dW = dD - (n * (dot3(dD, n) + dot3(d, dnv)) + dnv * dn) * 2.0f;
                } else {
                    const f3 nn = n * sig, dnn = dnv * sig;
                    const float dci = -(dot3(dD, nn) + dot3(d, dnn));
                    // (No renormalisation: the refracted direction of unit vectors is one.)
                    dW = dD * eta + nn * (dci * (eta - kd)) + dnn * (eta * ci - ct);
                }
                G.o[0][kp] = dP.x;
                G.o[1][kp] = dP.y;
                G.o[2][kp] = dP.z;
                G.d[0][kp] = dW.x;
                G.d[1][kp] = dW.y;
                G.d[2][kp] = dW.z;
            }
        }
        const bool last = k + 1 == L.count;
        o = mk3(q.x, q.y, last ? q.z + sf.z : q.z - sf.gap);
        oz = double(q.z) - sf.gapD;
        d = wv;
    }
    if (L.mirrors && obstructed(a, L, o, d, d.z > 0.0f ? __builtin_inff() : -__builtin_inff(), L.count - 1, L.count))
        return false;
    p = o;
    return d.z > 0.0f;
}

// The sums over a wave of N values per lane (N a power of two up to 32): lanes exchange halves of what they
// hold, so N + log2(64 / N) − 1 exchanges do what N separate sums take 6 N for. The sum of value j ends
// in v[0] of the lanes whose top log2(N) bits are j.
template <int N, int kHalf = N / 2>
__device__ __forceinline__ void waveSums(double (&v)[N], uint32_t lane) {
    if constexpr (kHalf >= 1) {
        constexpr int off = 64 * kHalf / N;
        const bool high = (lane & uint32_t(off)) != 0;
#pragma unroll
        for (int j = 0; j < kHalf; ++j) {
            const double give = high ? v[j] : v[j + kHalf], keep = high ? v[j + kHalf] : v[j];
            v[j] = keep + __shfl_xor(give, off);
        }
        waveSums<N, kHalf / 2>(v, lane);
    } else {
#pragma unroll
        for (int off = 32 / N; off >= 1; off /= 2) v[0] += __shfl_xor(v[0], off);
    }
}

// The block's bin table in LDS. Keys are bins of the lens the block is on (plane · pixels² + row ·
// pixels + column); a key is claimed by compare-and-swap, its sum grown by a 64-bit LDS add.
struct BinTable {
    uint32_t* keys;
    unsigned long long* sums;
};

// An add to LDS in the block's scope: with atomicAdd the compiler folds it and the add to HBM of a
// crowded table into one through a generic pointer, which is several times slower.
template <class V>
__device__ __forceinline__ void ldsAdd(V* p, V v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ uint32_t binSlot(uint32_t key) {
    static_assert(kHashSlots == 1 << 12, "the slot hash takes 12 bits");
    return (key * 2654435761u) >> (32 - 12);
}
// held: what the key's slot was last seen to hold. A claimed slot never changes before the flush, so
// a read (one for all lanes of a bin) finds most keys and only a first visitor swaps.
__device__ __forceinline__ void binAdd(BinTable t, unsigned long long* lensHist, uint32_t key, uint32_t held,
                                       unsigned long long v) {
    uint32_t slot = binSlot(key);
#pragma unroll 1
    for (int probe = 0; probe < kHashProbes; ++probe) {
        if (held == kHashEmpty) held = atomicCAS(&t.keys[slot], kHashEmpty, key);
        if (held == kHashEmpty || held == key) {
            ldsAdd(&t.sums[slot], v);
            return;
        }
        slot = (slot + 1) & uint32_t(kHashSlots - 1);
        held = t.keys[slot];
    }
    atomicAdd(lensHist + key, v);  // the table is crowded here: straight to HBM
}

// Adds every claimed bin of the table to the lens's grids and empties the table. By the whole block,
// between barriers.
__device__ __forceinline__ void binFlush(BinTable t, unsigned long long* lensHist) {
    for (uint32_t q = threadIdx.x; q < uint32_t(kHashSlots); q += kLensBlock) {
        const uint32_t key = t.keys[q];
        if (key != kHashEmpty) {
            atomicAdd(lensHist + key, t.sums[q]);
            t.keys[q] = kHashEmpty;
            t.sums[q] = 0;
        }
    }
}

// The persistent batch: a block takes the next `chunk` consecutive (lens, wavelength, block of rays)
// items, its threads trace each item's rays, the spot sums (and with kGrad the derivative sums of the
// pass's parameters) are reduced across each wave in double and added with one atomic each; grid
// adds go through the block's bin table, flushed when an item is another lens's and before the block
// exits. Chunks keep a block on one lens for most of its life, so few tables are flushed. Every
// barrier is reached by the whole block: items and their lens are uniform across it.
template <bool kGrad>
__global__ __launch_bounds__(kLensBlock) void lensKernel(LensArgs a) {
    __shared__ uint32_t tableKeys[kHashSlots];
    __shared__ unsigned long long tableSums[kHashSlots];
    __shared__ unsigned long long firstItem;
    const uint32_t lane = __lane_id();
    const bool sums = !kGrad || a.sums;
    const bool grids = sums && a.pixels > 0;
    const BinTable table{tableKeys, tableSums};
    if (grids)
        for (uint32_t q = threadIdx.x; q < uint32_t(kHashSlots); q += kLensBlock) {
            table.keys[q] = kHashEmpty;
            table.sums[q] = 0;
        }
    const size_t lensBins = size_t(a.planes) * a.pixels * a.pixels;
    uint32_t tableLens = ~0u;  // the lens whose bins the table holds
    uint64_t item = 0, lastItem = 0;
    for (;;) {
        if (item == lastItem) {
            __syncthreads();  // every thread has read the previous chunk's first item
            if (threadIdx.x == 0) firstItem = atomicAdd(a.next, (unsigned long long)a.chunk);
            __syncthreads();
            item = firstItem;
            // Uniform in scalar registers, so the lens's rows are read through the scalar unit.
            item = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(item)))) |
                   uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(item >> 32)))) << 32;
            lastItem = item + a.chunk;
        }
        if (item >= a.totalItems) break;
        // The lens of this item: the last whose first item is ≤ item.
        uint32_t lo = 0, len = a.nLenses;
        while (len > 0) {
            const uint32_t half = len / 2;
            if (a.lens[lo + half].itemBase <= item) {
                lo += half + 1;
                len -= half + 1;
            } else {
                len = half;
            }
        }
        const uint32_t li = lo - 1;
        const DLensInfo& L = a.lens[li];
        if (grids && li != tableLens) {
            __syncthreads();  // the table is clear, or every add of the previous lens is in it
            if (tableLens != ~0u) {
                binFlush(table, a.hist + tableLens * lensBins);
                __syncthreads();
            }
            tableLens = li;
        }
        unsigned long long* lensHist = a.hist + size_t(li) * lensBins;
        const uint64_t local = item - L.itemBase;
        ++item;
        const uint32_t w = uint32_t(local / L.itemsPerLambda);
        const uint64_t first = (local % L.itemsPerLambda) * a.raysPerItem;
        double m[OWE_LENS_MOMENTS - 1] = {0, 0, 0, 0, 0, 0, 0, 0};  // all but the count of arrived rays
        uint32_t arrived = 0;
        float gs[kGrad ? kGroup : 1][kGradSums] = {};
        for (uint32_t k = threadIdx.x; k < a.raysPerItem; k += kLensBlock) {
            const uint64_t i = first + k;
            if (i >= L.rays) break;
            f3 p, d;
            float T;
            RayGrad G;
            if (!traceLensRay<kGrad>(a, L, w, i, p, d, T, G)) continue;
            // The ray's spot terms in float (B = d_xy / d_z, A at z = 0 or the angles), summed in
            // double. An afocal spot's variance is 10⁻⁴ and less of its mean square, so its y angles
            // are taken relative to the angle refA of a slope refB near them, where float keeps their digits:
            // the argument of (1 + i b)(1 − i refB), in (−π, π), for a ray on either side of the axis.
            const float iz = quick(1.0f, d.z);
            const float bx = d.x * iz, by = d.y * iz;
            const float ax = L.afocal ? atanf(bx) : p.x - bx * p.z;
            const float ay = L.afocal ? atan2f(d.y - L.refB * d.z, d.z + L.refB * d.y) : p.y - by * p.z;
            if (kGrad) {
#pragma unroll
                for (int kp = 0; kp < kGroup; ++kp) {
                    const float dbx = (G.d[0][kp] * d.z - d.x * G.d[2][kp]) * iz * iz;
                    const float dby = (G.d[1][kp] * d.z - d.y * G.d[2][kp]) * iz * iz;
                    float dax, day;
                    if (L.afocal) {
                        dax = dbx / (1.0f + bx * bx);
                        day = dby / (1.0f + by * by);
                    } else {
                        dax = G.o[0][kp] - dbx * p.z - bx * G.o[2][kp];
                        day = G.o[1][kp] - dby * p.z - by * G.o[2][kp];
                    }
                    gs[kp][0] += dax;
                    gs[kp][1] += day;
                    gs[kp][2] += dbx;
                    gs[kp][3] += dby;
                    gs[kp][4] += ax * dax + ay * day;
                    gs[kp][5] += bx * dbx + by * dby;
                    gs[kp][6] += dax * bx + day * by + ax * dbx + ay * dby;
                }
            }
            if (!sums) continue;
            ++arrived;
            m[0] += double(ax);
            m[2] += double(bx);
            m[3] += double(by);
            if (L.afocal) {
                const double y = L.refA + double(ay);
                m[1] += y;
                m[4] += double(ax) * double(ax) + y * y;
                m[6] += double(ax) * double(bx) + y * double(by);
            } else {
                m[1] += double(ay);
                m[4] += double(ax * ax + ay * ay);
                m[6] += double(ax * bx + ay * by);
            }
            m[5] += double(bx * bx + by * by);
            m[7] += double(T);
            if (grids && L.detHalf > 0.0f) {
                const unsigned long long v = (unsigned long long)llrint(double(T) * kHistScale);
                const float half = 0.5f * float(a.planes - 1), mid = 0.5f * float(a.pixels);
                // Groups of planes: their table reads are in flight together.
                for (uint32_t first = 0; first < a.planes; first += kPlaneGroup) {
                    uint32_t key[kPlaneGroup], held[kPlaneGroup];
#pragma unroll
                    for (uint32_t g = 0; g < kPlaneGroup; ++g) {
                        key[g] = held[g] = kHashEmpty;
                        const uint32_t pl = first + g;
                        if (pl >= a.planes) continue;
                        const float s = L.detZ + (float(pl) - half) * L.detStep - p.z;
                        const float fx = mid + (p.x + bx * s - L.detX) * L.detScale;
                        const float fy = mid - (p.y + by * s - L.detY) * L.detScale;
                        if (!(fx >= 0.0f && fy >= 0.0f && fx < float(a.pixels) && fy < float(a.pixels))) continue;
                        const uint32_t px = min(uint32_t(fx), a.pixels - 1), py = min(uint32_t(fy), a.pixels - 1);
                        key[g] = (pl * a.pixels + py) * a.pixels + px;
                        held[g] = table.keys[binSlot(key[g])];
                    }
#pragma unroll
                    for (uint32_t g = 0; g < kPlaneGroup; ++g)
                        if (key[g] != kHashEmpty) binAdd(table, lensHist, key[g], held[g], v);
                }
            }
        }
        if (sums) {
            static_assert(OWE_LENS_MOMENTS == 9, "the arrived count and eight sums");
            double* dst = a.moments + (size_t(li) * a.nLambda + w) * OWE_LENS_MOMENTS;
            waveSums(m, lane);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) arrived += __shfl_xor(arrived, off);
            if (lane == 0 && arrived) atomicAdd(dst, double(arrived));
            if ((lane & 7u) == 0 && m[0] != 0.0) atomicAdd(dst + 1 + (lane >> 3), m[0]);
        }
        if (kGrad) {
            static_assert(kGroup * kGradSums <= 32, "a pass's derivative sums reduce together");
            double g[32] = {};
#pragma unroll
            for (int kp = 0; kp < kGroup; ++kp)
#pragma unroll
                for (int q = 0; q < kGradSums; ++q) g[kp * kGradSums + q] = double(gs[kp][q]);
            waveSums(g, lane);
            const uint32_t j = lane >> 1;
            if ((lane & 1u) == 0 && j < kGroup * kGradSums && a.paramBase + j / kGradSums < a.nParams && g[0] != 0.0)
                atomicAdd(a.grads + (size_t(li) * a.nLambda + w) * (OWE_LENS_MAX_PARAMS * kGradSums) +
                              a.paramBase * kGradSums + j, g[0]);
        }
    }
    __syncthreads();
    if (grids && tableLens != ~0u) binFlush(table, a.hist + tableLens * lensBins);
}

__global__ void lensBegin(LensArgs a, size_t nMoments, size_t nHist, size_t nGrads) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x, stride = size_t(gridDim.x) * blockDim.x;
    if (i == 0) *a.next = 0;
    for (size_t k = i; k < nMoments; k += stride) a.moments[k] = 0.0;
    for (size_t k = i; k < nHist; k += stride) a.hist[k] = 0;
    for (size_t k = i; k < nGrads; k += stride) a.grads[k] = 0.0;
}

// The irradiance grids from the weights' integers, each lens's scaled by its own factor. On the host the
// copy of 8-byte bins to pageable memory and their conversion took 12 ms of a 15 ms run with results
// (64 lenses, five planes of 128²); a float is all that leaves the card now, and that run takes 5.8 ms.
__global__ void lensResolve(const unsigned long long* hist, const double* scale, float* out, uint32_t lensBins, size_t first,
                            size_t n) {
    for (size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n; k += size_t(gridDim.x) * blockDim.x)
        out[k] = float(double(hist[first + k]) * scale[(first + k) / lensBins]);
}

// Resets the item counter between the gradient passes of one run.
__global__ void lensNext(LensArgs a) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.next = 0;
}

__global__ void lensProbe(LensArgs a, uint32_t li, uint32_t w, const uint64_t* index, uint64_t n, double* out) {
    const uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    f3 p, d;
    float T;
    RayGrad G;
    double* r = out + 7 * k;
    if (traceLensRay<false>(a, a.lens[li], w, index[k], p, d, T, G)) {
        r[0] = p.x, r[1] = p.y, r[2] = p.z, r[3] = d.x, r[4] = d.y, r[5] = d.z, r[6] = T;
    } else {
        for (int q = 0; q < 6; ++q) r[q] = __builtin_nan("");
        r[6] = 0.0;
    }
}

// ---------------------------------------------------------------- host: media and paraxial optics

double ciddor(double lnm) {
    const double s2 = (1e3 / lnm) * (1e3 / lnm);
    return 1 + 0.05792105 / (238.0185 - s2) + 0.00167917 / (57.362 - s2);
}
// IndexModel::n (src/owe/core/medium.cpp:46-66): absolute index, ×n_air when relative to air.
double mediumIndexHost(const owe_medium& m, double lnm) {
    const double l = lnm * 1e-3, l2 = l * l;
    double n = 1;
    switch (m.index_kind) {
        case OWE_INDEX_CONSTANT: n = m.coeff_a[0]; break;
        case OWE_INDEX_CAUCHY: n = m.coeff_a[0] + m.coeff_a[1] / l2 + m.coeff_a[2] / (l2 * l2); break;
        case OWE_INDEX_SELLMEIER: {
            double s = 1;
            for (int k = 0; k < m.terms; ++k) s += m.coeff_a[k] * l2 / (l2 - m.coeff_b[k]);
            n = std::sqrt(s);
            break;
        }
        case OWE_INDEX_CIDDOR: n = ciddor(lnm); break;
        default: fail(OWE_HIP_ERR_INVALID, "unknown index model");
    }
    return m.rel_air ? n * ciddor(lnm) : n;
}

struct ParaxialOut {
    double efl, bfl, epz, epr, length;
    double lastZ;  // the last vertex along the fixed chart (signed gaps)
    bool afocal;
    double angMag;
};

// paraxialAnalysis, object at infinity (src/owe/scene/prescription.cpp:193-321): the (y, n·u) system
// matrix with a refracting row's power (n' − n) c and a mirror's −2 dir n c (dir the travel along
// the fixed chart, which a mirror reverses; gaps unfolded), EFL −n'/C and BFL −n'A/C or — when C
// vanishes at the reference's scale — afocal with angular magnification D n/n', the stop (marked,
// else the surface that limits a marginal ray) and its image through the rows before it.
ParaxialOut paraxialHost(const owe_lens_surface* s, size_t N, const std::vector<double>& nAfter, double n0) {
    std::vector<double> nBefore(N), phi(N), t(N);
    double nPrev = n0, dir = 1;
    for (size_t i = 0; i < N; ++i) {
        nBefore[i] = nPrev;
        phi[i] = s[i].reflect ? -2 * dir * nAfter[i] * s[i].curvature : (nAfter[i] - nPrev) * s[i].curvature;
        if (s[i].reflect) dir = -dir;
        t[i] = std::fabs(s[i].thickness);
        nPrev = nAfter[i];
    }
    double a = 1, b = 0, c = 0, d = 1;
    for (size_t i = 0; i < N; ++i) {
        c -= phi[i] * a;
        d -= phi[i] * b;
        if (i + 1 < N) {
            const double k = t[i] / nAfter[i];
            a += k * c;
            b += k * d;
        }
    }
    ParaxialOut r{};
    for (size_t i = 0; i + 1 < N; ++i) {
        r.length += t[i];
        r.lastZ += s[i].thickness;
    }
    const double nk = nAfter[N - 1];
    const double scale = 1e-12 * (1 + std::fabs(a) + std::fabs(d));
    r.afocal = std::fabs(c) * std::max(1.0, r.length) < scale * 1e3 || std::fabs(c) < 1e-9;
    if (r.afocal) {
        r.efl = r.bfl = INFINITY;
        r.angMag = d * n0 / nk;
    } else {
        r.efl = -nk / c;
        r.bfl = -nk * a / c;
    }
    int stop = -1;
    for (size_t i = 0; i < N; ++i)
        if (s[i].stop) stop = int(i);
    if (stop < 0) {
        double best = -1, y = 1, nu = 0;
        for (size_t i = 0; i < N; ++i) {
            const double ratio = std::fabs(y) / std::max(s[i].semi_diameter, 1e-12);
            if (ratio > best) {
                best = ratio;
                stop = int(i);
            }
            nu -= phi[i] * y;
            if (i + 1 < N) y += t[i] * nu / nAfter[i];
        }
    }
    const double stopR = s[size_t(stop)].semi_diameter;
    double y = 0, nu = 1e-3 * nBefore[size_t(stop)], yM = stopR, nuM = 0;
    for (int i = stop - 1; i >= 0; --i) {
        y -= t[size_t(i)] * nu / nAfter[size_t(i)];
        yM -= t[size_t(i)] * nuM / nAfter[size_t(i)];
        nu += phi[size_t(i)] * y;
        nuM += phi[size_t(i)] * yM;
    }
    if (stop == 0) {
        r.epz = 0;
        r.epr = stopR;
    } else {
        const double u = nu / n0;
        require(u != 0, "entrance pupil at infinity");
        const double dz = -y / u;
        r.epz = dz;
        r.epr = std::fabs(yM + dz * nuM / n0);
    }
    return r;
}

}  // namespace
}  // namespace owehip

struct owe_hip_lens_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<void*> allocations;
    std::vector<owe_lens> lenses;
    std::vector<owe_lens_result> paraxial;  // launched/efl/bfl/pupil/last vertex per lens
    std::vector<DLensInfo> info;
    owe_lens_batch_settings settings{};
    LensArgs args{};
    size_t nMoments = 0, nHist = 0, nGrads = 0;
    double* gridScale = nullptr;    // irradiance per unit of a lens's bins (0: an afocal lens has no grid)
    float* irradiance = nullptr;    // up to kResolveBins of the grids on their way to the host
    int computeUnits = 256;
    int blocksPerCU = kResidentBlocks;
    hipEvent_t ev[2] = {nullptr, nullptr};
    double lastMs = 0;
    bool ran = false;
};

namespace owehip {
namespace {

template <class T>
T* lensAlloc(owe_hip_lens_batch* b, size_t n) {
    void* p = nullptr;
    OWE_HIP_CHECK(hipMalloc(&p, std::max<size_t>(1, n) * sizeof(T)));
    b->allocations.push_back(p);
    return static_cast<T*>(p);
}

// The grids become floats in pieces of up to 64 MiB, made with the batch: results cannot fail for memory after a
// run, and the largest batches need no second copy of their grids.
constexpr size_t kResolveBins = size_t(1) << 24;

// The work items of each lens of raysPerItem rays or, since a block traces an item, of the next whole number of
// rays to each of its threads: items of 64 rays would leave three waves of four idle (16 Gregorians with four
// derivatives 0.363 ms, with 256 rays 0.122; the form with an item to a wave 0.303 and 0.212).
void layoutItems(owe_hip_lens_batch* b, uint32_t raysPerItem) {
    raysPerItem = (raysPerItem + kLensBlock - 1) / kLensBlock * kLensBlock;
    uint64_t base = 0;
    for (DLensInfo& L : b->info) {
        L.itemBase = base;
        L.itemsPerLambda = uint32_t((L.rays + raysPerItem - 1) / raysPerItem);
        base += uint64_t(L.itemsPerLambda) * b->args.nLambda;
    }
    OWE_HIP_CHECK(hipMemcpy(const_cast<DLensInfo*>(b->args.lens), b->info.data(), b->info.size() * sizeof(DLensInfo),
                            hipMemcpyHostToDevice));
    b->args.raysPerItem = raysPerItem;
    b->args.totalItems = base;
}

// Rays per item before any tuning: eight items to each resident block, as a small batch needs every
// compute unit (256 rays, one to a thread) and a large one fewer reductions (4,096 rays).
uint32_t defaultItem(const owe_hip_lens_batch* b) {
    uint64_t rays = 0;
    for (const DLensInfo& L : b->info) rays += L.rays * b->args.nLambda;
    const uint64_t per = rays / (uint64_t(b->computeUnits) * uint64_t(kResidentBlocks) * 8);
    return uint32_t(std::clamp<uint64_t>((per + kLensBlock - 1) / kLensBlock * kLensBlock, kLensBlock, 4096));
}

// The chunk of items a block takes at a time: four chunks to a block of the grid, so blocks stay on a lens
// and the last chunks still even out.
uint32_t chunkOf(const owe_hip_lens_batch* b, unsigned blocks) {
    return uint32_t(std::clamp<uint64_t>(b->args.totalItems / (4 * uint64_t(blocks)), 1, 1u << 20));
}

// One run: the plain kernel, or with parameters set one gradient pass per kGroup parameters (the
// first also adding the spot sums and the histogram).
double runOnce(owe_hip_lens_batch* b) {
    hipLaunchKernelGGL(lensBegin, dim3{1024}, dim3{256}, 0, b->stream, b->args, b->nMoments, b->nHist, b->nGrads);
    OWE_HIP_CHECK(hipEventRecord(b->ev[0], b->stream));
    const dim3 grid{unsigned(std::max(1, b->computeUnits * b->blocksPerCU))};
    b->args.chunk = chunkOf(b, grid.x);
    if (b->args.nParams == 0) {
        hipLaunchKernelGGL(lensKernel<false>, grid, dim3{kLensBlock}, 0, b->stream, b->args);
    } else {
        for (uint32_t base = 0; base < b->args.nParams; base += kGroup) {
            LensArgs a = b->args;
            a.paramBase = base;
            a.sums = base == 0;
            if (base > 0) hipLaunchKernelGGL(lensNext, dim3{1}, dim3{64}, 0, b->stream, a);
            hipLaunchKernelGGL(lensKernel<true>, grid, dim3{kLensBlock}, 0, b->stream, a);
        }
    }
    OWE_HIP_CHECK(hipGetLastError());
    OWE_HIP_CHECK(hipEventRecord(b->ev[1], b->stream));
    OWE_HIP_CHECK(hipEventSynchronize(b->ev[1]));
    float ms = 0;
    OWE_HIP_CHECK(hipEventElapsedTime(&ms, b->ev[0], b->ev[1]));
    b->lastMs = ms;
    b->ran = true;
    return ms;
}

}  // namespace
}  // namespace owehip

extern "C" {

int owe_hip_lens_batch_create(int device, const owe_medium* media, uint32_t n_media, const owe_lens_surface* surfaces,
                              uint32_t n_surfaces, const owe_lens* lenses, uint32_t n_lenses,
                              const owe_lens_batch_settings* settings, owe_hip_lens_batch** out) {
    owe_hip_lens_batch* b = nullptr;
    const int st = guard([&] {
        require(out && media && surfaces && lenses && settings, "null argument");
        *out = nullptr;
        require(n_media > 0 && n_surfaces > 0 && n_lenses > 0, "empty batch");
        const owe_lens_batch_settings& s = *settings;
        require(s.n_wavelengths >= 1 && s.n_wavelengths <= OWE_LENS_MAX_WAVELENGTHS, "1 to 16 wavelengths");
        for (int w = 0; w < s.n_wavelengths; ++w)
            require(s.wavelengths[w] >= 300 && s.wavelengths[w] <= 2000, "wavelengths must lie in [300, 2000] nm");
        require(s.reference_wavelength >= 300 && s.reference_wavelength <= 2000, "reference wavelength out of range");
        require(std::fabs(s.field_deg) < 80, "field angle must lie in (-80, 80) degrees");
        require(s.detector_pixels >= 0 && s.detector_pixels <= 4096, "detector pixels must lie in [0, 4096]");
        require(s.detector_half_size >= 0, "detector half size must be non-negative");
        require(s.focus_planes >= 0 && s.focus_planes <= 16, "focus planes must lie in [0, 16]");
        require(s.focus_step >= 0 && std::isfinite(s.focus_step), "the focus step must be finite and non-negative");
        for (uint32_t i = 0; i < n_surfaces; ++i) {
            const owe_lens_surface& r = surfaces[i];
            const std::string name = "lens surface " + std::to_string(i);
            require(r.medium >= 0 && uint32_t(r.medium) < n_media, name + ": medium out of range");
            require(r.semi_diameter > 0 && std::isfinite(r.semi_diameter), name + ": semi-diameter must be positive");
            require(std::isfinite(r.curvature) && std::isfinite(r.conic) && std::isfinite(r.thickness),
                    name + ": values must be finite");
            require(1 - (1 + r.conic) * r.curvature * r.curvature * r.semi_diameter * r.semi_diameter >= 0,
                    name + ": aperture exceeds the domain of the conic");
            require(r.hole_radius >= 0 && (r.hole_radius == 0 || (r.reflect && r.hole_radius < r.semi_diameter)),
                    name + ": only a mirror has a hole, smaller than its semi-diameter");
        }
        selectDevice(device);
        b = new owe_hip_lens_batch;
        b->device = device;
        b->settings = s;
        hipDeviceProp_t prop;
        OWE_HIP_CHECK(hipGetDeviceProperties(&prop, device));
        b->computeUnits = prop.multiProcessorCount;
        OWE_HIP_CHECK(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
        OWE_HIP_CHECK(hipEventCreate(&b->ev[0]));
        OWE_HIP_CHECK(hipEventCreate(&b->ev[1]));
        const uint32_t nw = uint32_t(s.n_wavelengths);
        std::vector<DSurf> ds;
        std::vector<float> eta(size_t(n_surfaces) * nw, 1.0f);
        std::vector<uint8_t> used(n_surfaces, 0);
        // Lenses whose every root is polished in float64: instruments with mirrors or afocal ones,
        // where metre-long paths and the angular magnification turn a float root's error along
        // the ray (about 1e-7 of the path) into angular errors comparable to the spot itself.
        std::vector<uint8_t> precise;
        const double f = s.field_deg * 3.14159265358979323846 / 180;
        for (uint32_t li = 0; li < n_lenses; ++li) {
            const owe_lens& L = lenses[li];
            const std::string name = "lens " + std::to_string(li);
            require(L.surface_count >= 1 && uint64_t(L.first_surface) + L.surface_count <= n_surfaces,
                    name + ": surfaces out of range");
            require(L.rays >= 1 && L.rays <= (uint64_t(1) << 32), name + ": rays must lie in [1, 2^32]");
            require(L.ambient >= 0 && uint32_t(L.ambient) < n_media, name + ": ambient medium out of range");
            require(L.pupil_rings >= 0 && L.pupil_rings <= 30000, name + ": pupil rings must lie in [0, 30000]");
            require(L.pupil_rings == 0 || L.rays == 1 + 3 * uint64_t(L.pupil_rings) * uint64_t(L.pupil_rings + 1),
                    name + ": with pupil rings r the lens traces 1 + 3 r (r + 1) rays");
            const owe_lens_surface* rows = surfaces + L.first_surface;
            std::vector<double> nRef(L.surface_count);
            int mirrors = 0;
            uint64_t mirrorMask = 0;
            for (uint32_t k = 0; k < L.surface_count; ++k) {
                require(!used[L.first_surface + k], name + ": surfaces are shared with another lens");
                used[L.first_surface + k] = 1;
                if (rows[k].reflect) {
                    ++mirrors;
                    if (k < 64) mirrorMask |= uint64_t(1) << k;
                    require(rows[k].medium == (k == 0 ? L.ambient : rows[k - 1].medium),
                            name + ": a mirror reflects into the medium it is met in");
                }
                nRef[k] = mediumIndexHost(media[rows[k].medium], s.reference_wavelength);
                const owe_medium& before = media[k == 0 ? L.ambient : rows[k - 1].medium];
                for (uint32_t w = 0; w < nw; ++w)
                    eta[size_t(L.first_surface + k) * nw + w] =
                        float(mediumIndexHost(before, s.wavelengths[w]) / mediumIndexHost(media[rows[k].medium], s.wavelengths[w]));
            }
            const ParaxialOut px = paraxialHost(rows, L.surface_count, nRef, mediumIndexHost(media[L.ambient], s.reference_wavelength));
            owe_lens_result r{};
            r.launched = L.rays * nw;
            r.efl = px.efl;
            r.bfl = px.bfl;
            r.entrance_pupil_z = px.epz;
            r.entrance_pupil_radius = px.epr;
            r.last_vertex_z = px.lastZ;
            r.afocal = px.afocal ? 1 : 0;
            r.angular_magnification = px.angMag;
            b->paraxial.push_back(r);
            DLensInfo I{};
            I.first = L.first_surface;
            I.count = L.surface_count;
            I.rays = L.rays;
            I.rings = uint32_t(L.pupil_rings);
            I.rEP = px.epr;
            I.zEP = px.epz;
            I.zStart = -0.05 - 0.1 * px.length;
            I.yStart = std::sin(f) * ((I.zStart - I.zEP) / std::cos(f));
            // The detector: the paraxial image plane at the reference wavelength, centred on the
            // chief ray's paraxial image height EFL·tan θ.
            I.detZ = float(px.lastZ + px.bfl);
            I.detX = 0.0f;
            I.detY = float(px.efl * std::tan(f));
            I.detHalf = float(s.detector_half_size > 0 ? s.detector_half_size : 5e-3 * std::fabs(px.efl));
            I.detStep = float(s.focus_step > 0 ? s.focus_step : 1e-3 * std::fabs(px.efl));
            I.afocal = px.afocal ? 1 : 0;
            I.mirrors = mirrors;
            I.mirrorMask = mirrorMask;
            I.refB = px.afocal ? float(px.angMag * std::tan(f)) : 0.0f;
            I.refA = std::atan(double(I.refB));
            if (px.afocal) {  // no image plane: no irradiance grid
                I.detZ = I.detY = I.detHalf = I.detStep = 0.0f;
            }
            I.detScale = I.detHalf > 0 ? float(0.5 * s.detector_pixels / double(I.detHalf)) : 0.0f;
            b->info.push_back(I);
            precise.push_back(mirrors > 0 || px.afocal);
        }
        ds.resize(n_surfaces);
        for (uint32_t li = 0; li < n_lenses; ++li) {
            const owe_lens& L = lenses[li];
            double z = 0;
            for (uint32_t k = 0; k < L.surface_count; ++k) {
                const owe_lens_surface& r = surfaces[L.first_surface + k];
                DSurf d{};
                static_cast<DSag&>(d) = makeSag(r.curvature, r.conic, r.asphere, r.semi_diameter,
                                                r.reflect ? r.hole_radius : 0.0);
                d.polish64 = precise[li] || std::fabs(r.curvature) * r.semi_diameter > kSteepPolish ? 1 : 0;
                d.z = float(z);
                d.gap = float(r.thickness);
                d.gapD = r.thickness;
                d.reflect = r.reflect ? 1 : 0;
                ds[L.first_surface + k] = d;
                z += r.thickness;
            }
        }
        b->lenses.assign(lenses, lenses + n_lenses);
        LensArgs& a = b->args;
        DSurf* dsurf = lensAlloc<DSurf>(b, ds.size());
        OWE_HIP_CHECK(hipMemcpy(dsurf, ds.data(), ds.size() * sizeof(DSurf), hipMemcpyHostToDevice));
        a.surf = dsurf;
        a.lens = lensAlloc<DLensInfo>(b, n_lenses);
        float* de = lensAlloc<float>(b, eta.size());
        OWE_HIP_CHECK(hipMemcpy(de, eta.data(), eta.size() * sizeof(float), hipMemcpyHostToDevice));
        a.eta = de;
        a.nLenses = n_lenses;
        a.nLambda = nw;
        a.pixels = uint32_t(s.detector_pixels);
        a.planes = uint32_t(std::max(1, s.focus_planes));
        a.dirY = std::sin(f);
        a.dirZ = std::cos(f);
        a.next = lensAlloc<unsigned long long>(b, 1);
        b->nMoments = size_t(n_lenses) * nw * OWE_LENS_MOMENTS;
        a.moments = lensAlloc<double>(b, b->nMoments);
        b->nHist = size_t(n_lenses) * a.planes * a.pixels * a.pixels;
        a.hist = lensAlloc<unsigned long long>(b, b->nHist);
        if (b->nHist > 0) {
            // Unit irradiance across the beam: each ray carries π r² cos θ / (rays · nλ) of flux.
            std::vector<double> scale(n_lenses, 0.0);
            for (uint32_t li = 0; li < n_lenses; ++li) {
                const DLensInfo& I = b->info[li];
                if (!(I.detHalf > 0)) continue;
                const double pix = 2.0 * I.detHalf / a.pixels;
                scale[li] = 3.14159265358979323846 * I.rEP * I.rEP * 0.999 * 0.999 * a.dirZ /
                            (double(I.rays) * nw * kHistScale * pix * pix);
            }
            b->gridScale = lensAlloc<double>(b, n_lenses);
            OWE_HIP_CHECK(hipMemcpy(b->gridScale, scale.data(), n_lenses * sizeof(double), hipMemcpyHostToDevice));
            b->irradiance = lensAlloc<float>(b, std::min(b->nHist, kResolveBins));
        }
        b->nGrads = 0;
        a.grads = lensAlloc<double>(b, size_t(n_lenses) * nw * OWE_LENS_MAX_PARAMS * kGradSums);
        a.nParams = 0;
        layoutItems(b, defaultItem(b));
        *out = b;
    });
    if (st != OWE_HIP_OK && b) {
        for (void* p : b->allocations) (void)hipFree(p);
        for (hipEvent_t e : b->ev)
            if (e) (void)hipEventDestroy(e);
        if (b->stream) (void)hipStreamDestroy(b->stream);
        delete b;
    }
    return st;
}

int owe_hip_lens_batch_destroy(owe_hip_lens_batch* b) {
    return guard([&] {
        if (!b) return;
        (void)hipSetDevice(b->device);
        if (b->stream) (void)hipStreamSynchronize(b->stream);
        for (void* p : b->allocations) OWE_HIP_CHECK(hipFree(p));
        for (hipEvent_t e : b->ev)
            if (e) OWE_HIP_CHECK(hipEventDestroy(e));
        if (b->stream) OWE_HIP_CHECK(hipStreamDestroy(b->stream));
        delete b;
    });
}

int owe_hip_lens_batch_run(owe_hip_lens_batch* b) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        OWE_HIP_CHECK(hipSetDevice(b->device));
        runOnce(b);
    });
}

int owe_hip_lens_batch_set_params(owe_hip_lens_batch* b, const owe_lens_param* params, uint32_t n) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        require(n <= OWE_LENS_MAX_PARAMS, "at most OWE_LENS_MAX_PARAMS parameters");
        require(n == 0 || params != nullptr, "null parameters");
        uint32_t minCount = ~0u;
        for (const owe_lens& L : b->lenses) minCount = std::min(minCount, L.surface_count);
        for (uint32_t k = 0; k < n; ++k) {
            require(params[k].surface < minCount, "parameter surface beyond a lens's surfaces");
            require(params[k].field >= OWE_LENS_PARAM_CURVATURE && params[k].field <= OWE_LENS_PARAM_A4 + 3,
                    "unknown parameter field");
            b->args.paramSurface[k] = int32_t(params[k].surface);
            b->args.paramField[k] = params[k].field;
        }
        b->args.nParams = n;
        b->nGrads = n ? size_t(b->lenses.size()) * b->args.nLambda * OWE_LENS_MAX_PARAMS * kGradSums : 0;
        b->ran = false;
    });
}

int owe_hip_lens_batch_gradients(owe_hip_lens_batch* b, double* grad) {
    return guard([&] {
        require(b != nullptr && grad != nullptr, "null argument");
        require(b->ran, "run the batch first");
        require(b->args.nParams > 0, "no parameters are set");
        const size_t nl = b->lenses.size(), nw = b->args.nLambda, np = b->args.nParams;
        std::vector<double> mom(nl * nw * OWE_LENS_MOMENTS), gs(nl * nw * OWE_LENS_MAX_PARAMS * kGradSums);
        OWE_HIP_CHECK(hipMemcpy(mom.data(), b->args.moments, mom.size() * sizeof(double), hipMemcpyDeviceToHost));
        OWE_HIP_CHECK(hipMemcpy(gs.data(), b->args.grads, gs.size() * sizeof(double), hipMemcpyDeviceToHost));
        for (size_t li = 0; li < nl; ++li) {
            double m[OWE_LENS_MOMENTS] = {};
            std::vector<double> g(np * kGradSums, 0.0);
            for (size_t w = 0; w < nw; ++w) {
                for (int q = 0; q < OWE_LENS_MOMENTS; ++q) m[q] += mom[(li * nw + w) * OWE_LENS_MOMENTS + q];
                for (size_t k = 0; k < np * kGradSums; ++k) g[k] += gs[(li * nw + w) * OWE_LENS_MAX_PARAMS * kGradSums + k];
            }
            const double n = m[0];
            for (size_t k = 0; k < np; ++k) {
                double out = NAN;
                // ΣA'x, ΣA'y, ΣB'x, ΣB'y, ΣA·A', ΣB·B', Σ(A'·B + A·B'); afocal: A relative to (0, refA).
                const double* G = &g[k * kGradSums];
                if (n >= 3) {
                    const double max = m[1] / n, may = m[2] / n, mbx = m[3] / n, mby = m[4] / n;
                    const double dmax = G[0] / n, dmay = G[1] / n, dmbx = G[2] / n, dmby = G[3] / n;
                    if (b->paraxial[li].afocal) {
                        // v = Σ|A|²/n − 2 c·ΣA/n + |c|², c = atan(mean B): afocalSpot's RMS².
                        const double cx = std::atan(mbx), cy = std::atan(mby);
                        const double dcx = dmbx / (1 + mbx * mbx), dcy = dmby / (1 + mby * mby);
                        const double v = m[5] / n - 2 * (cx * max + cy * may) + cx * cx + cy * cy;
                        // v' = 2 E[(A − c)·A'] − 2 c'·(E A − c).
                        const double ref = b->info[li].refA;
                        const double dv = 2 * (G[4] / n - cx * dmax + (ref - cy) * dmay) -
                                          2 * (dcx * (max - cx) + dcy * (may - cy));
                        out = v > 0 ? dv / (2 * std::sqrt(v)) : 0.0;
                    } else {
                        // rms² at best focus = var_A − cov²/var_B (focusedSpot).
                        const double va = m[5] / n - (max * max + may * may);
                        const double vb = m[6] / n - (mbx * mbx + mby * mby);
                        const double cv = m[7] / n - (max * mbx + may * mby);
                        const double dva = 2 * G[4] / n - 2 * (max * dmax + may * dmay);
                        const double dvb = 2 * G[5] / n - 2 * (mbx * dmbx + mby * dmby);
                        const double dcv = G[6] / n - (dmax * mbx + dmay * mby + max * dmbx + may * dmby);
                        const double r2 = vb > 0 ? va - cv * cv / vb : va;
                        const double dr2 = vb > 0 ? dva - (2 * cv * dcv * vb - cv * cv * dvb) / (vb * vb) : dva;
                        out = r2 > 0 ? dr2 / (2 * std::sqrt(r2)) : 0.0;
                    }
                }
                grad[li * np + k] = out;
            }
        }
    });
}

int owe_hip_lens_batch_last_ms(const owe_hip_lens_batch* b, double* ms) {
    return guard([&] {
        require(b != nullptr && ms != nullptr, "null argument");
        *ms = b->lastMs;
    });
}

int owe_hip_lens_batch_set_shape(owe_hip_lens_batch* b, int blocks_per_cu, int rays_per_item) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        require(blocks_per_cu >= 0 && blocks_per_cu <= 64, "blocks per compute unit must lie in [0, 64]");
        require(rays_per_item >= 0 && rays_per_item % 64 == 0 && rays_per_item <= (1 << 20),
                "rays per item must be a multiple of 64 up to 2^20");
        OWE_HIP_CHECK(hipSetDevice(b->device));
        if (blocks_per_cu > 0) b->blocksPerCU = blocks_per_cu;
        if (rays_per_item > 0) layoutItems(b, uint32_t(rays_per_item));
    });
}

int owe_hip_lens_batch_autotune(owe_hip_lens_batch* b, double* best_ms) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        OWE_HIP_CHECK(hipSetDevice(b->device));
        // Every shape is timed once; the three fastest three more times each, and the lowest median
        // wins, so one noisy run cannot pick the shape.
        struct Cand {
            int blocks;
            uint32_t rays;
            double ms;
        };
        std::vector<Cand> cands;
        auto run = [&](const Cand& c) {
            b->blocksPerCU = c.blocks;
            layoutItems(b, c.rays);
            return runOnce(b);
        };
        // Up to the resident blocks, and grids of more, whose chunks are smaller (chunkOf): 256 achromats take 15.1 ms
        // with eight blocks and 19.1 with three, 48 achromats 1.02 with three, four and eight, six small lenses 0.021 with
        // two and 0.037 with eight. And the batch's own item.
        std::vector<uint32_t> items{256u, 1024u, 4096u, 16384u};
        const uint32_t own = defaultItem(b);
        if (std::find(items.begin(), items.end(), own) == items.end()) items.push_back(own);
        for (int blocks : {1, 2, kResidentBlocks, 4, 8})
            for (uint32_t rays : items) {
                cands.push_back({blocks, rays, 0.0});
                cands.back().ms = run(cands.back());
            }
        std::sort(cands.begin(), cands.end(), [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
        for (size_t i = 0; i < 3 && i < cands.size(); ++i) {
            double t[3];
            for (double& x : t) x = run(cands[i]);
            std::sort(t, t + 3);
            cands[i].ms = t[1];
        }
        std::sort(cands.begin(), cands.begin() + std::min<size_t>(3, cands.size()),
                  [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
        const double best = cands.front().ms;
        b->blocksPerCU = cands.front().blocks;
        layoutItems(b, cands.front().rays);
        b->ran = false;
        if (best_ms) *best_ms = best;
    });
}

int owe_hip_lens_batch_results(owe_hip_lens_batch* b, owe_lens_result* lenses, double* moments, float* irradiance) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        require(b->ran, "no run yet");
        OWE_HIP_CHECK(hipSetDevice(b->device));
        const uint32_t nl = uint32_t(b->lenses.size()), nw = b->args.nLambda, px = b->args.pixels;
        std::vector<double> m(b->nMoments);
        OWE_HIP_CHECK(hipMemcpy(m.data(), b->args.moments, m.size() * sizeof(double), hipMemcpyDeviceToHost));
        if (moments) std::copy(m.begin(), m.end(), moments);
        if (lenses) {
            for (uint32_t li = 0; li < nl; ++li) {
                owe_lens_result r = b->paraxial[li];
                double s[OWE_LENS_MOMENTS] = {0};
                for (uint32_t w = 0; w < nw; ++w)
                    for (int q = 0; q < OWE_LENS_MOMENTS; ++q) s[q] += m[(size_t(li) * nw + w) * OWE_LENS_MOMENTS + q];
                r.arrived = uint64_t(s[0]);
                r.transmitted = s[8] / double(r.launched);
                // focusedSpot (analysis.cpp:85-113) from the sums, or afocalSpot (70-81) from the
                // sums of angles.
                const double zImg = r.last_vertex_z + r.bfl;
                r.apparent_angle = r.angular_rms = NAN;
                if (r.afocal) {
                    r.best_focus_z = r.rms_best = r.rms_paraxial = r.centroid_y = NAN;
                    if (s[0] >= 3) {
                        const double n = s[0], cx = std::atan(s[3] / n), cy = std::atan(s[4] / n);
                        const double v = s[5] / n - 2 * (cx * s[1] + cy * s[2]) / n + cx * cx + cy * cy;
                        r.apparent_angle = cy;
                        r.angular_rms = std::sqrt(std::max(0.0, v));
                    }
                } else if (s[0] >= 3) {
                    const double n = s[0], max_ = s[1] / n, may = s[2] / n, mbx = s[3] / n, mby = s[4] / n;
                    const double varA = s[5] / n - (max_ * max_ + may * may), varB = s[6] / n - (mbx * mbx + mby * mby);
                    const double cov = s[7] / n - (max_ * mbx + may * mby);
                    const double zBest = varB > 0 ? -cov / varB : zImg;
                    auto rms = [&](double z) { return std::sqrt(std::max(0.0, varA + 2 * z * cov + z * z * varB)); };
                    r.best_focus_z = zBest - r.last_vertex_z;
                    r.rms_best = rms(zBest);
                    r.rms_paraxial = rms(zImg);
                    r.centroid_y = may + mby * zImg;
                } else {
                    r.best_focus_z = r.rms_best = r.rms_paraxial = r.centroid_y = NAN;
                }
                lenses[li] = r;
            }
        }
        if (irradiance && px > 0) {
            for (size_t at = 0; at < b->nHist; at += kResolveBins) {
                const size_t n = std::min(kResolveBins, b->nHist - at);
                hipLaunchKernelGGL(lensResolve, dim3{2048}, dim3{256}, 0, b->stream, b->args.hist, b->gridScale,
                                   b->irradiance, uint32_t(b->args.planes * px * px), at, n);
                OWE_HIP_CHECK(hipGetLastError());
                OWE_HIP_CHECK(hipMemcpyAsync(irradiance + at, b->irradiance, n * sizeof(float), hipMemcpyDeviceToHost, b->stream));
                OWE_HIP_CHECK(hipStreamSynchronize(b->stream));
            }
        }
    });
}

int owe_hip_lens_batch_trace(owe_hip_lens_batch* b, uint32_t lens, int wavelength, const uint64_t* index, uint64_t n,
                             double* out) {
    return guard([&] {
        require(b != nullptr, "batch is null");
        require(lens < b->lenses.size(), "lens out of range");
        require(wavelength >= 0 && uint32_t(wavelength) < b->args.nLambda, "wavelength out of range");
        if (n == 0) return;
        require(index != nullptr && out != nullptr, "null buffer");
        for (uint64_t k = 0; k < n; ++k) require(index[k] < b->lenses[lens].rays, "ray index out of range");
        OWE_HIP_CHECK(hipSetDevice(b->device));
        uint64_t* di = nullptr;
        double* dout = nullptr;
        OWE_HIP_CHECK(hipMalloc(&di, n * sizeof(uint64_t)));
        OWE_HIP_CHECK(hipMalloc(&dout, 7 * n * sizeof(double)));
        OWE_HIP_CHECK(hipMemcpy(di, index, n * sizeof(uint64_t), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(lensProbe, dim3{unsigned((n + 255) / 256)}, dim3{256}, 0, b->stream, b->args, lens,
                           uint32_t(wavelength), di, n, dout);
        const hipError_t e = hipGetLastError();
        if (e == hipSuccess) {
            (void)hipStreamSynchronize(b->stream);
            (void)hipMemcpy(out, dout, 7 * n * sizeof(double), hipMemcpyDeviceToHost);
        }
        (void)hipFree(di);
        (void)hipFree(dout);
        OWE_HIP_CHECK(e);
    });
}

}  // extern "C"
