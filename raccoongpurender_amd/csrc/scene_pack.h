// Device side of rgpu_scene_create (scene_pack.hip): the tables the kernels read, packed on the
// GPU from the host's tree and geometry.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bvh_build.h"
#include "rgpu_traverse.h"

namespace rgpu {

// Device allocations of a scene; each may be null (nothing of its kind).
struct SceneTables {
    void* walk = nullptr;
    void* prims = nullptr;
    void* points = nullptr;
    void* indices = nullptr;
    void* spheres = nullptr;
};

// Uploads the tree and the geometry and packs the walk records (the first kTreeletMaxNodes in
// breadth-first order, so that any LDS copy of the top of the tree is a prefix, the others in the
// tree's depth-first order), the primitive records and the float4 vertices on stream s, and fills
// dev. Synchronous. On an error what was allocated is left in *tables for the caller to free.
hipError_t pack_scene(const BVHTree& t, const float* points, uint32_t stride, uint32_t npoints,
                      const uint32_t* indices, uint32_t ntris, const float* spheres, uint32_t nspheres, hipStream_t s,
                      SceneTables* tables, TraceScene* dev);

}  // namespace rgpu
