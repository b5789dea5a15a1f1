// pt_gpu.h -- device-resident builders shared by the renderer and the unit entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "pt_internal.h"
#include "pt_types.h"

namespace pt {

#define PT_HIP_TRY(expr)                                                                   \
    do {                                                                                   \
        hipError_t _e = (expr);                                                            \
        if (_e != hipSuccess) {                                                            \
            throw HipFailure(std::string(#expr) + ": " + hipGetErrorString(_e));           \
        }                                                                                  \
    } while (0)

struct HipFailure {
    std::string msg;
    explicit HipFailure(std::string m) : msg(std::move(m)) {}
};

// Owning device allocation (hipMalloc / hipFree).
struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    void alloc(size_t n) {
        if (n == bytes && p) return;
        release();
        if (n == 0) return;
        PT_HIP_TRY(hipMalloc(&p, n));
        bytes = n;
    }
    template <class T> T *as() const { return (T *)p; }
};

// One device allocation cut into several arrays (a hipMalloc and a hipFree cost as much as a
// kernel each).  want() notes the pointers, alloc() sets them.
struct WorkArrays {
    struct Want {
        void **p;
        size_t bytes;
    };
    std::vector<Want> wants;
    DevBuf buf;
    template <class T> void want(T *&p, size_t n) { wants.push_back({(void **)&p, (n * sizeof(T) + 255) / 256 * 256}); }
    void alloc() {
        std::vector<Want> now;
        now.swap(wants);   // also where there is no memory for them
        size_t total = 256;
        for (const Want &w : now) total += w.bytes;
        buf.alloc(total);
        size_t at = 0;
        for (const Want &w : now) {
            *w.p = buf.as<char>() + at;
            at += w.bytes;
        }
    }
};

// Copies device memory to pageable host memory behind the stream's work and waits for it: through
// pinned staging memory, a piece copied out by the CPU while the next ones are on the link.
void readToHost(void *dst, const void *src, size_t bytes, hipStream_t stream);

// An int of pinned host memory that kernels can write, from a page shared by the process's
// objects (pinning memory for each costs 100 us); null when the page is used up.
class HostWord {
public:
    HostWord();
    ~HostWord();
    HostWord(const HostWord &) = delete;
    HostWord &operator=(const HostWord &) = delete;
    int *p = nullptr;
};

// An int that a kernel writes and the host reads once the stream is idle.
class HostInt {
public:
    int *target() {
        if (!word.p) own.alloc(sizeof(int));
        return word.p ? word.p : own.as<int>();
    }
    int read() const {
        int v = 0;
        if (word.p) v = *(volatile int *)word.p;
        else PT_HIP_TRY(hipMemcpy(&v, own.p, sizeof v, hipMemcpyDeviceToHost));
        return v;
    }

private:
    HostWord word;
    DevBuf own;   // where no pinned word was to be had
};

struct BvhInfo {
    int numNodes = 0;      // 4-wide nodes
    int depth = 0;         // levels of 4-wide nodes
    int binaryDepth = 0;   // levels of internal nodes of the binary radix tree
};

// Binary-tree builders of buildBvh.
enum { PT_BVH_LBVH = 0, PT_BVH_PLOC = 1 };

// Builds a binary BVH over `n` primitive records (3 float4 each, input order) on `stream`
// (builder: PT_BVH_LBVH or PT_BVH_PLOC) and collapses it into a 4-wide BVH on the GPU:
// allocates `nodes` (PT_NODE_F4 float4 per node) and writes the records in BVH order to
// `primsSorted`.  lo/hi bound all primitive centroids.
void buildBvh(const float4 *primsIn, int n, const float lo[3], const float hi[3], DevBuf &nodes,
              float4 *primsSorted, hipStream_t stream, BvhInfo *info, int builder);

// Environment tables in FP64 on the GPU: per-row and marginal alias tables packed as
// (prob as float, alias as int bits), texel pdf.  Optionally returns the FP64 tables.
void buildEnvTables(const float4 *rgba, int w, int h, int sinWeight, float2 *rows, float2 *marginal,
                    float *texelPdf, double *rowProbOut, int *rowAliasOut, double *margProbOut,
                    int *margAliasOut, hipStream_t stream);

// Copies the texel pdf into the w component of the environment texels (PtEnv::rgba).
void packEnvPdf(float4 *rgba, const float *texelPdf, int n, hipStream_t stream);

int deviceCUs();

// Exclusive prefix sums of m counters in place, the total to data[m] (m + 1 entries); tmp holds
// scanEntries(m).
size_t scanEntries(int m);
void scanCounts(uint32_t *data, int m, uint32_t *tmp, hipStream_t stream);

// The scene's arrays on the device as the host describes them, in input order, and the device
// records made from them.  Kept for edits: a material changes in place, and an emission edit
// makes the emitter list again.
struct SceneArrays {
    int nTri = 0, nSph = 0, nMat = 0;
    WorkArrays arrays;
    float *pos = nullptr, *sph = nullptr;   // 9 per triangle, 4 per sphere
    int *triMat = nullptr, *sphMat = nullptr;
    HostMaterial *mats = nullptr;
    // Uploads s and writes its primitive records (triangles, then spheres), the per-vertex
    // normals that differ from the flat ones, and the bounds (+-infinity without primitives).
    void load(const pt_scene &s, DevBuf &records, DevBuf &normals, float lo[3], float hi[3], hipStream_t stream);
    void buildMaterials(DevBuf &records, hipStream_t stream) const;
    // Emitter records (3 float4 each) in the reference's light order; returns their number.
    int buildEmitters(DevBuf &records, HostInt &answer, hipStream_t stream) const;
    // A material's new values, in place; null colours stay.  The emitters' number: they are listed again
    // where the material is emissive now or was.
    int editMaterial(int id, int type, const float *albedo, const float *emit, float ior, float alpha, DevBuf &materials, DevBuf &emitters,
                     int emittersNow, HostInt &answer, hipStream_t stream);
};

}  // namespace pt
