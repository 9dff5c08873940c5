// Batch ray queries on a triangle mesh: the C-ABI owe_hip_mesh_* and owe_hip_trace_batch.
// Stands in for MeshShape::intersect over many rays (src/owe/scene/mesh.cpp:73-97) and the float
// kernels' any-hit occludedMesh (src/owe/backends/gpu/shaders/geometry.slang:577-615).
//
// One kernel (traceKernel) of persistent waves, each owning a contiguous range of rays: a lane whose
// ray has ended waits until `refill` lanes of its wave are idle; then those write their results and
// take the next rays of the range together. The form of one lane per ray is the same kernel with 64
// rays to a wave. Per step a wave either visits a node or tests triangles, two a lane at most, in all the lanes that are
// at one (traverse.hpp): a ray meets a leaf in one node of eight, so testing the leaves of a node where
// it is visited, as the transport kernels' traverseBvh4 does, ran the triangle test with 1 to 5 lanes
// of 64. Near two limits at once: 10.2 GB beyond L2 for 8,388,608 closest queries on 1,048,820 triangles (90 MB of
// nodes and triangles against 4 MiB of L2 per XCD) at the rate of a large copy, and VALU busy 91 % of the time with half
// of the lanes. Launches back to back: 4.02 → 1.90 ms closest and 3.05 → 1.46 ms any hit; 0.48 → 0.27 and
// 0.35 → 0.19 ms for 1,000,003 rays on 100,820 triangles. 4,096 rays on 20,480 triangles take 33 µs closest and 28 any
// hit, as before: the longest ray's chain of loads (the host's call is 7 µs, and waiting for it adds 15).
#include <hip/hip_runtime.h>

#include <string>

#include "bvh4.hpp"
#include "common.hpp"
#include "traverse.hpp"

using namespace owehip;

struct owe_hip_mesh {
    int device = 0;
    WideNode* nodes = nullptr;
    TriRecord* tris = nullptr;
    owe_hip_mesh_stats stats{};
    int cus = 0;                 // compute units of the device
    // Per query mode (closest, any): the launch form, and the refill form's resident blocks per
    // compute unit and idle lanes that trigger a refill.
    int form[2] = {OWE_HIP_TRACE_REFILL, OWE_HIP_TRACE_REFILL};
    int blocksPerCu[2] = {8, 8};
    int refill[2] = {32, 32};
};

namespace owehip {
namespace {

constexpr int kQueryBlock = 128;

// Wave w owns rays [w·per, min(n, (w + 1)·per)). Every branch that decides a refill or the step's kind is
// wave-uniform (ballots and the range); no barrier is used, so waves run independently and each exits
// once its range is drained and its lanes are idle. Results are written at a refill, many lanes
// at once; lanes end out of order, so the lines fill in a few partial writes that L2 gathers.
// The triangle step runs when the lanes at a leaf are half as many as those at a node, or when none is at
// a node: of thresholds from a quarter to one and a half, and of fixed counts from 1 to 32, this one
// was the fastest closest query (2.0 ms with one triangle a step; 8 lanes fixed 2.4, 24 lanes fixed 2.3) and none was faster for any hit.
template <bool kAny>
__global__ __launch_bounds__(kQueryBlock) void traceKernel(const WideNode* __restrict__ nodes,
                                                           const TriRecord* __restrict__ tris,
                                                           const float4* __restrict__ rays, uint64_t n, uint64_t per,
                                                           uint32_t refill, uint32_t* __restrict__ primOut,
                                                           float* __restrict__ tOut) {
    __shared__ uint32_t stack[kWalkLds * kQueryBlock];
    uint32_t mem[kWalkStack - kWalkLds];
    const WalkStack st{stack + threadIdx.x, mem};
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kQueryBlock / 64) + (threadIdx.x >> 6));
    uint64_t next = wave * per;
    const uint64_t end = next < n ? (n - next < per ? n : next + per) : next;
    constexpr uint64_t kNoRay = ~0ull;
    uint64_t ray = kNoRay;  // the ray of this lane whose result is not written yet
    Walk s;
    s.hit.slot = s.cur = kEmptyChild;
    for (;;) {
        const bool idle = s.cur == kEmptyChild;
        const uint64_t idleMask = __ballot(idle);
        const uint32_t nIdle = uint32_t(__popcll(idleMask));
        if (nIdle == 64u || (next < end && nIdle >= refill)) {
            if (idle && ray != kNoRay) {
                const bool miss = s.hit.slot == kEmptyChild;
                primOut[ray] = miss ? 0xFFFFFFFFu : tris[s.hit.slot].prim;
                tOut[ray] = miss ? __builtin_inff() : s.hit.t;
                ray = kNoRay;
            }
            if (next >= end) break;
            const uint32_t rank = uint32_t(__popcll(idleMask & ((1ull << lane) - 1ull)));
            if (idle && next + rank < end) {
                ray = next + rank;
                const float4 r0 = rays[2 * ray], r1 = rays[2 * ray + 1];
                walkBegin(s, mk3(r0.x, r0.y, r0.z), mk3(r1.x, r1.y, r1.z), r0.w, r1.w);
            }
            next = end - next > nIdle ? next + nIdle : end;
        }
        const bool active = s.cur != kEmptyChild;
        const bool atLeaf = active && (s.cur & kLeafBit) != 0;
        const uint32_t leaves = uint32_t(__popcll(__ballot(atLeaf)));
        const uint32_t inner = uint32_t(__popcll(__ballot(active && !atLeaf)));
        if (2 * leaves >= inner) {
            if (atLeaf) walkTriangle<kAny>(s, tris, st, kQueryBlock);
        } else {
            if (active && !atLeaf) walkNode(s, nodes, st, kQueryBlock);
        }
    }
}

void launchTrace(int mode, const owe_hip_mesh* m, const float* rays, uint64_t n, uint32_t* prim, float* t,
                 hipStream_t s) {
    const int q = mode == OWE_HIP_QUERY_ANY ? 1 : 0;
    constexpr uint64_t kWaves = kQueryBlock / 64;
    uint64_t blocks, per = 64;
    uint32_t refill = 64;
    if (m->form[q] == OWE_HIP_TRACE_REFILL) {
        blocks = uint64_t(m->cus) * uint64_t(m->blocksPerCu[q]);
        per = (n + blocks * kWaves - 1) / (blocks * kWaves);
        refill = uint32_t(m->refill[q]);
    } else {
        blocks = (n + kQueryBlock - 1) / kQueryBlock;
        if (blocks > 0x7FFFFFFFull) fail(OWE_HIP_ERR_INVALID, "batch too large for one launch");
    }
    const dim3 grid{unsigned(blocks)}, block{unsigned(kQueryBlock)};
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, m->nodes, m->tris, reinterpret_cast<const float4*>(rays), n, per,
                           refill, prim, t);
    };
    if (mode == OWE_HIP_QUERY_ANY) go(traceKernel<true>);
    else go(traceKernel<false>);
    OWE_HIP_CHECK(hipGetLastError());
}

}  // namespace
}  // namespace owehip

extern "C" {

int owe_hip_mesh_create(int device, const float* positions, uint32_t nVertices, const uint32_t* triangles,
                        uint32_t nTriangles, owe_hip_mesh** out) {
    return guard([&] {
        require(out != nullptr, "out is null");
        require(positions != nullptr || nVertices == 0, "positions is null");
        require(triangles != nullptr || nTriangles == 0, "triangles is null");
        *out = nullptr;
        selectDevice(device);
        Bvh4 b = buildBvh4(positions, nVertices, triangles, nTriangles);
        if (b.stackBound > 64)
            fail(OWE_HIP_ERR_UNSUPPORTED, "mesh hierarchy needs a traversal stack of " + std::to_string(b.stackBound) +
                                              " entries; the kernels hold at most 64");
        auto* m = new owe_hip_mesh;
        m->device = device;
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, device) != hipSuccess || prop.multiProcessorCount <= 0) {
            delete m;
            fail(OWE_HIP_ERR_DEVICE, "cannot read the device's compute-unit count");
        }
        m->cus = prop.multiProcessorCount;
        const size_t nb = b.nodes.size() * sizeof(WideNode), tb = std::max<size_t>(1, b.tris.size()) * sizeof(TriRecord);
        hipError_t e = hipMalloc(&m->nodes, nb);
        if (e == hipSuccess) e = hipMalloc(&m->tris, tb);
        if (e == hipSuccess) e = hipMemcpy(m->nodes, b.nodes.data(), nb, hipMemcpyHostToDevice);
        if (e == hipSuccess && !b.tris.empty())
            e = hipMemcpy(m->tris, b.tris.data(), b.tris.size() * sizeof(TriRecord), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            if (m->nodes) (void)hipFree(m->nodes);
            if (m->tris) (void)hipFree(m->tris);
            delete m;
            hipCheck(e, "mesh upload");
        }
        m->stats.triangles = nTriangles;
        m->stats.nodes = b.nodes.size();
        m->stats.depth = b.depth;
        m->stats.stack_bound = b.stackBound;
        m->stats.build_seconds = b.seconds;
        m->stats.device_bytes = nb + tb;
        *out = m;
    });
}

int owe_hip_mesh_destroy(owe_hip_mesh* m) {
    return guard([&] {
        if (!m) return;
        (void)hipSetDevice(m->device);
        if (m->nodes) OWE_HIP_CHECK(hipFree(m->nodes));
        if (m->tris) OWE_HIP_CHECK(hipFree(m->tris));
        delete m;
    });
}

int owe_hip_mesh_stats_get(const owe_hip_mesh* m, owe_hip_mesh_stats* out) {
    return guard([&] {
        require(m != nullptr && out != nullptr, "null argument");
        *out = m->stats;
    });
}

int owe_hip_mesh_set_launch(owe_hip_mesh* m, int mode, int form, int blocks_per_cu, int refill) {
    return guard([&] {
        require(m != nullptr, "mesh is null");
        require(mode == -1 || mode == OWE_HIP_QUERY_CLOSEST || mode == OWE_HIP_QUERY_ANY,
                "mode must be closest (0), any (1) or both (-1)");
        require(form == OWE_HIP_TRACE_PER_LANE || form == OWE_HIP_TRACE_REFILL, "form must be 0 (per lane) or 1 (refill)");
        require(blocks_per_cu >= 0 && blocks_per_cu <= 10, "blocks_per_cu must be 0 (keep) to 10");
        require(refill >= 0 && refill <= 64, "refill must be 0 (keep) to 64");
        for (int q = 0; q < 2; ++q) {
            if (mode != -1 && mode != q) continue;
            m->form[q] = form;
            if (blocks_per_cu) m->blocksPerCu[q] = blocks_per_cu;
            if (refill) m->refill[q] = refill;
        }
    });
}

int owe_hip_mesh_get_launch(const owe_hip_mesh* m, int mode, int* form, int* blocks_per_cu, int* refill) {
    return guard([&] {
        require(m != nullptr && form != nullptr && blocks_per_cu != nullptr && refill != nullptr, "null argument");
        require(mode == OWE_HIP_QUERY_CLOSEST || mode == OWE_HIP_QUERY_ANY, "mode must be closest (0) or any (1)");
        *form = m->form[mode];
        *blocks_per_cu = m->blocksPerCu[mode];
        *refill = m->refill[mode];
    });
}

int owe_hip_trace_batch(owe_hip_mesh* m, int mode, const float* rays, uint64_t n, uint32_t* prim, float* t,
                        void* stream) {
    return guard([&] {
        require(m != nullptr, "mesh is null");
        require(mode == OWE_HIP_QUERY_CLOSEST || mode == OWE_HIP_QUERY_ANY, "mode must be closest (0) or any (1)");
        if (n == 0) return;
        require(rays != nullptr && prim != nullptr && t != nullptr, "null buffer");
        require((reinterpret_cast<uintptr_t>(rays) & 15) == 0, "rays must be 16-byte aligned");
        for (const void* p : {static_cast<const void*>(rays), static_cast<const void*>(prim), static_cast<const void*>(t)}) {
            hipPointerAttribute_t a;
            if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice || a.device != m->device)
                fail(OWE_HIP_ERR_INVALID, "rays, prim and t must be device memory on the mesh's device");
        }
        OWE_HIP_CHECK(hipSetDevice(m->device));
        const hipStream_t s = static_cast<hipStream_t>(stream);
        launchTrace(mode, m, rays, n, prim, t, s);
    });
}

}  // extern "C"
