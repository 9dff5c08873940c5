// Per-lane traversal of the 4-wide BVH (bvh4.hpp) for one ray: closest hit or any hit.
//
// Semantics follow the reference's mesh query (src/owe/scene/mesh.cpp:73-97 over
// src/owe/scene/bvh.hpp:31-78): a triangle counts when the line crosses it (watertight test) and its
// plane distance t lies strictly inside (tmin, best); the closest wins. The slab test keeps the
// reference float kernels' conservative far bound (shaders/geometry.slang:398-416): widened by a few
// ulps so rounding never culls a box the triangle test would hit.
//
// gfx950 layout: every lane walks its own ray. A node visit is one 128-byte line (eight 16-byte
// loads). Hit leaf children are intersected at once, nearest inner child is entered next, and the
// other hit inner children go on a short stack in LDS laid out [entry][lane] so a wave's pushes and
// pops touch 64 consecutive banks. The stack's capacity is the build's exact bound, so it never
// overflows.
#pragma once

#include "bvh4.hpp"
#include "dmath.hpp"

namespace owehip {

struct RayHit {
    float t;
    uint32_t slot;  // triangle record index (leaf order), kEmptyChild on a miss
};

// skipFace: a spawned ray's own face (its coplanar triangles are not crossings); ~0u for none.
// stack: this lane's first entry in LDS; stride: lanes per block.
// Contacts (world queries only; a triangle record's last word names its boundary): triangles of
// boundary `own` count from tmin, those of every other boundary from tminOther (below zero for a
// spawned ray: a touching surface at its origin); skipFace2 is a second face group that is skipped.
template <bool kAny>
__device__ inline RayHit traverseBvh4(const WideNode* __restrict__ nodes, const TriRecord* __restrict__ tris, f3 o, f3 d,
                                      float tmin, float tmax, uint32_t skipFace, uint32_t* stack, uint32_t stride,
                                      uint32_t own = ~0u, float tminOther = 0.0f, uint32_t skipFace2 = ~0u) {
    const bool contact = own != ~0u;
    const float tlow = contact ? fminf(tmin, tminOther) : tmin;
    const Shear sh = makeShear(d);
    const f3 inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    const bool nx = inv.x < 0.0f, ny = inv.y < 0.0f, nz = inv.z < 0.0f;
    RayHit hit{tmax, kEmptyChild};
    uint32_t sp = 0;
    uint32_t cur = 0;
    for (;;) {
        const float4* q = reinterpret_cast<const float4*>(nodes + cur);
        const float4 lx = q[0], hx = q[1], ly = q[2], hy = q[3], lz = q[4], hz = q[5];
        const uint4 ch = reinterpret_cast<const uint4*>(nodes + cur)[6];
        const float lxs[4] = {lx.x, lx.y, lx.z, lx.w}, hxs[4] = {hx.x, hx.y, hx.z, hx.w};
        const float lys[4] = {ly.x, ly.y, ly.z, ly.w}, hys[4] = {hy.x, hy.y, hy.z, hy.w};
        const float lzs[4] = {lz.x, lz.y, lz.z, lz.w}, hzs[4] = {hz.x, hz.y, hz.z, hz.w};
        const uint32_t cs[4] = {ch.x, ch.y, ch.z, ch.w};
        float tn[4];
        bool hitc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float x0 = ((nx ? hxs[c] : lxs[c]) - o.x) * inv.x, x1 = ((nx ? lxs[c] : hxs[c]) - o.x) * inv.x;
            const float y0 = ((ny ? hys[c] : lys[c]) - o.y) * inv.y, y1 = ((ny ? lys[c] : hys[c]) - o.y) * inv.y;
            const float z0 = ((nz ? hzs[c] : lzs[c]) - o.z) * inv.z, z1 = ((nz ? lzs[c] : hzs[c]) - o.z) * inv.z;
            const float near = fmaxf(fmaxf(tlow, x0), fmaxf(y0, z0));
            float far = fminf(fminf(x1, y1), z1);
            far = far * (far >= 0.0f ? 1.0000004f : 0.9999996f);
            far = fminf(far, hit.t);
            tn[c] = near;
            hitc[c] = near <= far;
        }
        // Leaf children now, in slot order; inner children by entry distance (static indexing only,
        // so the candidates stay in registers).
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (!hitc[c] || !(cs[c] & kLeafBit)) continue;
            const uint32_t first = cs[c] & kFirstMask, count = ((cs[c] >> kCountShift) & 0xFu) + 1;
            for (uint32_t k = 0; k < count; ++k) {
                const uint32_t slot = first + k;
                const float4* tr = reinterpret_cast<const float4*>(tris + slot);
                const float4 a = tr[0], b = tr[1], cc = tr[2];
                if (skipFace != ~0u && __float_as_uint(b.w) == skipFace) continue;
                if (skipFace2 != ~0u && __float_as_uint(b.w) == skipFace2) continue;
                const float tl = contact && __float_as_uint(cc.w) != own ? tminOther : tmin;
                float t;
                if (!hitTriangle(sh, o, d, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), mk3(cc.x, cc.y, cc.z), tl, hit.t, t))
                    continue;
                hit.t = t;
                hit.slot = slot;
                if (kAny) return hit;
            }
        }
        // Inner children still nearer than the closest hit found so far.
        float key[4];
        uint32_t nd[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool inner = hitc[c] && !(cs[c] & kLeafBit) && tn[c] <= hit.t;
            key[c] = inner ? tn[c] : __builtin_inff();
            nd[c] = inner ? cs[c] : kEmptyChild;
        }
        // Four-key sorting network: (0,1) (2,3) (0,2) (1,3) (1,2).
        auto order = [&](int i, int j) {
            if (key[j] < key[i]) {
                const float tk = key[i];
                key[i] = key[j];
                key[j] = tk;
                const uint32_t tn2 = nd[i];
                nd[i] = nd[j];
                nd[j] = tn2;
            }
        };
        order(0, 1);
        order(2, 3);
        order(0, 2);
        order(1, 3);
        order(1, 2);
        // Empty entries sorted last (key +inf); an inner child entered at +inf sorts among them but
        // keeps its node index, so validity is the index, not the key.
#pragma unroll
        for (int k = 3; k >= 1; --k)
            if (nd[k] != kEmptyChild) stack[(sp++) * stride] = nd[k];
        if (nd[0] != kEmptyChild) {
            cur = nd[0];
            continue;
        }
        if (sp == 0) break;
        cur = stack[(--sp) * stride];
    }
    return hit;
}

// The walk of batch ray queries (rayquery.hip) in single steps, so that a kernel can choose for a
// whole wave whether it visits nodes or tests triangles next. A lane's position is `cur`: a node, a
// leaf reference whose first triangle comes next, or kEmptyChild once its ray has ended. A visited
// node's children go on the stack, inner ones far to near, then the leaves it hits in reverse slot
// order, and the top is entered next; what a ray visits, and in which order, depends on the ray
// alone and not on its wave. Culling happens when a node is visited: keeping each entry's distance to
// cull it when popped saves a fifth of a closest query's visits (13.4 of 16.6 on the 1,048,820-triangle
// mesh) but its longer pops cost more than that (2.33 against 2.0 ms for 8,388,608 rays, one triangle a step).
struct Walk {
    f3 o, d, inv;
    Shear sh;
    float tmin;
    RayHit hit;
    uint32_t sp, cur;
    uint32_t nearX, nearY, nearZ;  // byte offsets of a node's near planes; the far ones are 16 away
};

// The lower kWalkLds entries of a lane's stack lie in LDS as [entry][lane], the others, which few
// rays reach, in private memory: 16 entries let as many waves in as the registers do. A visit leaves
// at most four entries more than the build's bound on inner nodes, plus one slot that is written
// but not kept.
constexpr uint32_t kWalkLds = 16;
constexpr uint32_t kWalkStack = 64 + 5;  // the mesh queries' largest bound
struct WalkStack {
    uint32_t* lds;  // this lane's first entry; entries are `stride` apart
    uint32_t* mem;  // kWalkStack − kWalkLds private entries
};

__device__ __forceinline__ void walkBegin(Walk& w, f3 o, f3 d, float tmin, float tmax) {
    w.o = o;
    w.d = d;
    w.sh = makeShear(d);
    w.inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    w.nearX = w.inv.x < 0.0f ? 16u : 0u;
    w.nearY = w.inv.y < 0.0f ? 48u : 32u;
    w.nearZ = w.inv.z < 0.0f ? 80u : 64u;
    w.tmin = tmin;
    w.hit = RayHit{tmax, kEmptyChild};
    w.sp = 0;
    w.cur = 0;
}

__device__ __forceinline__ void walkPop(Walk& w, const WalkStack& st, uint32_t stride) {
    if (w.sp == 0) {
        w.cur = kEmptyChild;
        return;
    }
    --w.sp;
    w.cur = w.sp < kWalkLds ? st.lds[w.sp * stride] : st.mem[w.sp - kWalkLds];
}

// Visits node w.cur. The planes are loaded as near and far ones by the ray's signs, so no selects
// follow. far + |far| · 3·2⁻²³ is the slab's widened far bound (traverseBvh4's factor for far ≥ 0);
// an empty child has far = −inf, which it turns into NaN: no comparison accepts it.
__device__ __forceinline__ void walkNode(Walk& w, const WideNode* __restrict__ nodes, const WalkStack& st, uint32_t stride) {
    const char* p = reinterpret_cast<const char*>(nodes + w.cur);
    auto planes = [&](uint32_t at) { return *reinterpret_cast<const float4*>(p + at); };
    const float4 nx = planes(w.nearX), fx = planes(w.nearX ^ 16u);
    const float4 ny = planes(w.nearY), fy = planes(w.nearY ^ 16u);
    const float4 nz = planes(w.nearZ), fz = planes(w.nearZ ^ 16u);
    const uint4 ch = reinterpret_cast<const uint4*>(p)[6];
    const float nxs[4] = {nx.x, nx.y, nx.z, nx.w}, fxs[4] = {fx.x, fx.y, fx.z, fx.w};
    const float nys[4] = {ny.x, ny.y, ny.z, ny.w}, fys[4] = {fy.x, fy.y, fy.z, fy.w};
    const float nzs[4] = {nz.x, nz.y, nz.z, nz.w}, fzs[4] = {fz.x, fz.y, fz.z, fz.w};
    const uint32_t cs[4] = {ch.x, ch.y, ch.z, ch.w};
    float key[4];
    uint32_t nd[4];
    bool leaf[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float x0 = (nxs[c] - w.o.x) * w.inv.x, x1 = (fxs[c] - w.o.x) * w.inv.x;
        const float y0 = (nys[c] - w.o.y) * w.inv.y, y1 = (fys[c] - w.o.y) * w.inv.y;
        const float z0 = (nzs[c] - w.o.z) * w.inv.z, z1 = (fzs[c] - w.o.z) * w.inv.z;
        const float near = fmaxf(fmaxf(fmaxf(w.tmin, x0), y0), z0);
        const float far = fminf(fminf(x1, y1), z1);
        const bool met = near <= __builtin_fmaf(fabsf(far), 0x1.8p-22f, far) && near <= w.hit.t;
        const bool isLeaf = (cs[c] & kLeafBit) != 0;
        leaf[c] = met && isLeaf;
        key[c] = met && !isLeaf ? near : __builtin_inff();
        nd[c] = met && !isLeaf ? cs[c] : kEmptyChild;
    }
    // Four-key sorting network, as traverseBvh4's.
    auto order = [&](int i, int j) {
        if (key[j] < key[i]) {
            const float tk = key[i];
            key[i] = key[j];
            key[j] = tk;
            const uint32_t tn = nd[i];
            nd[i] = nd[j];
            nd[j] = tn;
        }
    };
    order(0, 1);
    order(2, 3);
    order(0, 2);
    order(1, 3);
    order(1, 2);
    const bool anyLeaf = leaf[0] || leaf[1] || leaf[2] || leaf[3];
    if (__ballot(w.sp + 9 > kWalkLds) == 0) {
        // Room in LDS for the whole wave: every entry is written, the ones that count move the top.
        uint32_t* top = st.lds + w.sp * stride;
        auto push = [&](bool keep, uint32_t ref) {
            *top = ref;
            top += keep ? stride : 0u;
            w.sp += keep ? 1u : 0u;
        };
#pragma unroll
        for (int k = 3; k >= 1; --k) push(nd[k] != kEmptyChild, nd[k]);
        if (__ballot(anyLeaf) == 0) {  // no lane met a leaf: the nearest inner child needs no stack
            w.cur = nd[0];
            if (w.cur == kEmptyChild) walkPop(w, st, stride);
            return;
        }
        push(nd[0] != kEmptyChild, nd[0]);
#pragma unroll
        for (int c = 3; c >= 0; --c) push(leaf[c], cs[c]);
    } else {
        auto push = [&](bool keep, uint32_t ref) {
            if (!keep) return;
            if (w.sp < kWalkLds) st.lds[w.sp * stride] = ref;
            else st.mem[w.sp - kWalkLds] = ref;
            ++w.sp;
        };
#pragma unroll
        for (int k = 3; k >= 0; --k) push(nd[k] != kEmptyChild, nd[k]);
#pragma unroll
        for (int c = 3; c >= 0; --c) push(leaf[c], cs[c]);
    }
    walkPop(w, st, stride);
}

// Tests the first two triangles of leaf reference w.cur (its only one where it has one) and moves to its next
// ones, or to the stack's top. Both are loaded together: one wait for two tests, where one triangle a step
// took 2.0 ms for 8,388,608 closest queries and 0.207 for 1,000,003 any-hit ones (with two 1.9 and 0.199; 4,096 queries
// take the same with either).
template <bool kAny>
__device__ __forceinline__ void walkTriangle(Walk& w, const TriRecord* __restrict__ tris, const WalkStack& st,
                                             uint32_t stride) {
    constexpr int kMost = 2;
    float4 v[kMost][3];
    const uint32_t slot = w.cur & kFirstMask, more = (w.cur >> kCountShift) & 0xFu;  // triangles behind the first
    const float4* tr = reinterpret_cast<const float4*>(tris + slot);
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        const uint32_t at = uint32_t(k) <= more ? uint32_t(k) : 0u;
#pragma unroll
        for (int i = 0; i < 3; ++i) v[k][i] = tr[3 * at + i];
    }
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        float t;
        const f3 p0 = mk3(v[k][0].x, v[k][0].y, v[k][0].z), p1 = mk3(v[k][1].x, v[k][1].y, v[k][1].z),
                 p2 = mk3(v[k][2].x, v[k][2].y, v[k][2].z);
        if (uint32_t(k) <= more && hitTriangle(w.sh, w.o, w.d, p0, p1, p2, w.tmin, w.hit.t, t)) {
            w.hit = RayHit{t, slot + uint32_t(k)};
            if (kAny) {
                w.cur = kEmptyChild;
                return;
            }
        }
    }
    if (more >= uint32_t(kMost)) w.cur += uint32_t(kMost) * (1u - (1u << kCountShift));  // fewer triangles, from a later slot
    else walkPop(w, st, stride);
}

}  // namespace owehip
