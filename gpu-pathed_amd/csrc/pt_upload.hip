// pt_upload.hip -- host arrays to the device and images back.
//
// A scene upload copies positions, material ids, spheres and materials to the device unchanged
// and builds the 48-byte primitive records, the 32-byte material records, the scene bounds, the
// per-vertex normals worth keeping and the emitter list there.  What bounds it is the copy over
// the host link (80 B per triangle of a scene with per-face materials).  Making the records on
// the host wrote and faulted in another 170 B per triangle of fresh host memory for one pass of
// trivial work: 1.31M triangles with per-face materials took 43 ms on the host before, beside
// 21 ms of kernels.
#include <hip/hip_runtime.h>

#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <memory>
#include <mutex>
#include <thread>

#include "pt_gpu.h"
#include "pt_internal.h"

namespace pt {

namespace {

constexpr int kThreads = 256;
constexpr int kBoundsBlocks = 512;
inline unsigned blocksOf(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kThreads - 1) / kThreads); }

__global__ __launch_bounds__(kThreads) void k_upload_prims(const float *pos, const int *triMat, const uint32_t *normalAt, const uint32_t *smooth, int nt,
                                                           const float *sph, const int *sphMat, int ns, float4 *recs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nt) {
        const float *p = pos + 9 * (size_t)i;
        // smooth triangles point at their three normals, in order
        const int tag = smooth && smooth[i] ? (int)normalAt[i] : PT_TAG_FLAT;
        recs[3 * (size_t)i] = make_float4(p[0], p[1], p[2], asFloat(triMat[i]));
        recs[3 * (size_t)i + 1] = make_float4(p[3], p[4], p[5], asFloat(tag));
        recs[3 * (size_t)i + 2] = make_float4(p[6], p[7], p[8], asFloat(i));
    } else if (i < nt + ns) {
        const int k = i - nt;
        const float *q = sph + 4 * (size_t)k;
        recs[3 * (size_t)i] = make_float4(q[0], q[1], q[2], asFloat(sphMat[k]));
        recs[3 * (size_t)i + 1] = make_float4(q[3], 0.f, 0.f, asFloat(PT_TAG_SPHERE));
        recs[3 * (size_t)i + 2] = make_float4(0.f, 0.f, 0.f, asFloat(~k));
    }
}

// Bounds of the records' vertices and sphere centres: a box per block, then one block's fold.
__device__ __forceinline__ void blockBounds(float lo[3], float hi[3], float *out) {
    __shared__ float part[kThreads / 64][6];
    for (int k = 0; k < 3; k++)
        for (int off = 32; off >= 1; off >>= 1) {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], off));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], off));
        }
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; k++) {
            part[threadIdx.x >> 6][k] = lo[k];
            part[threadIdx.x >> 6][3 + k] = hi[k];
        }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; k++) {
            float v = part[0][k];
            for (int w = 1; w < kThreads / 64; w++) v = k < 3 ? fminf(v, part[w][k]) : fmaxf(v, part[w][k]);
            out[k] = v;
        }
}

__global__ __launch_bounds__(kThreads) void k_bounds(const float4 *recs, int n, float *boxes) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    auto grow = [&](float4 v) {
        const float c[3] = {v.x, v.y, v.z};
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], c[k]);
            hi[k] = fmaxf(hi[k], c[k]);
        }
    };
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float4 a = recs[3 * (size_t)i], b = recs[3 * (size_t)i + 1], c = recs[3 * (size_t)i + 2];
        grow(a);
        if (asInt(b.w) != PT_TAG_SPHERE) {
            grow(b);
            grow(c);
        }
    }
    blockBounds(lo, hi, boxes + 6 * blockIdx.x);
}

__global__ __launch_bounds__(kThreads) void k_bounds_fold(const float *boxes, int n, float *out) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], boxes[6 * i + k]);
            hi[k] = fmaxf(hi[k], boxes[6 * i + 3 + k]);
        }
    blockBounds(lo, hi, out);
}

// 1 where a triangle's per-vertex normals differ from its flat one (only those are kept).
__global__ __launch_bounds__(kThreads) void k_smooth_flags(const float *pos, const float *nrm, int nt, uint32_t *smooth, uint32_t *rank) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    const float *p = pos + 9 * (size_t)i, *nv = nrm + 9 * (size_t)i;
    const float e1[3] = {p[3] - p[0], p[4] - p[1], p[5] - p[2]}, e2[3] = {p[6] - p[0], p[7] - p[1], p[8] - p[2]};
    const float g[3] = {e1[1] * e2[2] - e1[2] * e2[1], -(e1[0] * e2[2] - e1[2] * e2[0]), e1[0] * e2[1] - e1[1] * e2[0]};
    const float gl = sqrtf(g[0] * g[0] + g[1] * g[1] + g[2] * g[2]);
    bool flat = gl > 0.f;
    for (int v = 0; v < 3; v++)
        for (int k = 0; k < 3; k++)
            if (fabsf(nv[v * 3 + k] - g[k] / gl) > 1e-6f) flat = false;
    smooth[i] = flat ? 0u : 1u;
    rank[i] = flat ? 0u : 1u;
}

__global__ __launch_bounds__(kThreads) void k_keep_normals(const float *nrm, const uint32_t *smooth, const uint32_t *rank, int nt, float4 *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt || !smooth[i]) return;
    const float *nv = nrm + 9 * (size_t)i;
    for (int v = 0; v < 3; v++) out[3 * (size_t)rank[i] + v] = make_float4(nv[3 * v], nv[3 * v + 1], nv[3 * v + 2], 0.f);
}

// Emission is a Lambertian's alone (params.h:37-70).
__device__ __forceinline__ bool emits(const HostMaterial &m) {
    return m.type == PT_LAMBERTIAN && (m.emit[0] != 0.f || m.emit[1] != 0.f || m.emit[2] != 0.f);
}

__device__ __forceinline__ void writeMaterial(const HostMaterial &h, PtMaterial *out) {
    const bool lamb = h.type == PT_LAMBERTIAN;
    const float param = h.type == PT_GLASS ? h.ior : (h.type == PT_MICROFACET ? h.alpha : 0.f);
    out->a = make_float4(h.albedo[0], h.albedo[1], h.albedo[2], (float)h.type);
    out->b = make_float4(lamb ? h.emit[0] : 0.f, lamb ? h.emit[1] : 0.f, lamb ? h.emit[2] : 0.f, param);
}

__global__ __launch_bounds__(kThreads) void k_materials(const HostMaterial *mats, int n, PtMaterial *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) writeMaterial(mats[i], &out[i]);
}

// An edit of one material: the kept one and its record, or of id -1 none.  True where it was or is
// emissive.
struct MaterialEdit {
    int id = -1, setAlbedo = 0, setEmit = 0;
    HostMaterial to{};
};
__device__ __forceinline__ bool applyEdit(const MaterialEdit &e, HostMaterial *mats, PtMaterial *records) {
    const HostMaterial was = mats[e.id];
    HostMaterial to = e.to;
    for (int k = 0; k < 3; k++) {
        if (!e.setAlbedo) to.albedo[k] = was.albedo[k];
        if (!e.setEmit) to.emit[k] = was.emit[k];
    }
    mats[e.id] = to;
    writeMaterial(to, &records[e.id]);
    return emits(was) || emits(to);
}

// The host waits for what it needs to know, which this writes to pinned memory: reading the material back,
// changing it and copying it up again took 37 us a call, this 15.
__global__ void k_edit_material(MaterialEdit e, HostMaterial *mats, PtMaterial *records, int *emissive) {
    if (threadIdx.x == 0) *emissive = applyEdit(e, mats, records) ? 1 : 0;
}

__global__ __launch_bounds__(kThreads) void k_emitter_flags(const HostMaterial *mats, const int *triMat, int nt, const int *sphMat, int ns,
                                                            uint32_t *rank) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt + ns) return;
    rank[i] = emits(mats[i < nt ? triMat[i] : sphMat[i - nt]]) ? 1u : 0u;
}

// Emitter records in the reference light order (scene_data.cu:92-115): emissive triangles by
// index, then emissive spheres.  Their normals are the flat ones.
__device__ __forceinline__ void writeEmitter(const float *pos, const int *triMat, int nt, const float *sph, const int *sphMat, int i, float4 *o) {
    if (i < nt) {
        const float *p = pos + 9 * (size_t)i;
        o[0] = make_float4(p[0], p[1], p[2], asFloat(triMat[i]));
        o[1] = make_float4(p[3], p[4], p[5], asFloat(PT_TAG_FLAT));
        o[2] = make_float4(p[6], p[7], p[8], asFloat(i));
    } else {
        const int k = i - nt;
        const float *s = sph + 4 * (size_t)k;
        o[0] = make_float4(s[0], s[1], s[2], asFloat(sphMat[k]));
        o[1] = make_float4(s[3], 0.f, 0.f, asFloat(PT_TAG_SPHERE));
        o[2] = make_float4(0.f, 0.f, 0.f, asFloat(~k));
    }
}

__global__ __launch_bounds__(kThreads) void k_emitters(const HostMaterial *mats, const float *pos, const int *triMat, int nt, const float *sph,
                                                       const int *sphMat, int ns, const uint32_t *rank, float4 *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt + ns) return;
    if (emits(mats[i < nt ? triMat[i] : sphMat[i - nt]])) writeEmitter(pos, triMat, nt, sph, sphMat, i, out + 3 * (size_t)rank[i]);
}

// The list by one block, and its length, for scenes of up to kEmittersSmall primitives, after an edit or
// without one; an edit that has nothing to do with emission leaves the list of `now` emitters.  Flags,
// prefix sums, the length's way to the host and the records' allocation took half of an emission edit's
// 74 us; with the edit in the same launch it takes 16.
constexpr int kEmittersSmall = 2048;
constexpr int kEmittersThreads = 1024;
__global__ __launch_bounds__(kEmittersThreads) void k_emitters_small(MaterialEdit e, HostMaterial *mats, PtMaterial *records, const float *pos,
                                                                     const int *triMat, int nt, const float *sph, const int *sphMat, int ns, int now,
                                                                     float4 *out, int *count) {
    __shared__ int sWave[kEmittersThreads / 64], sList;
    if (threadIdx.x == 0) sList = e.id < 0 || applyEdit(e, mats, records) ? 1 : 0;
    __syncthreads();
    if (sList == 0) {
        if (threadIdx.x == 0) *count = now;
        return;
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int base = 0;
    for (int i0 = 0; i0 < nt + ns; i0 += kEmittersThreads) {
        const int i = i0 + threadIdx.x;
        const bool mine = i < nt + ns && emits(mats[i < nt ? triMat[i] : sphMat[i - nt]]);
        const uint64_t m = __ballot(mine);
        if (lane == 0) sWave[wave] = __popcll(m);
        __syncthreads();
        int at = base + __popcll(m & ((1ull << lane) - 1));
        for (int w = 0; w < kEmittersThreads / 64; w++) {
            if (w < wave) at += sWave[w];
            base += sWave[w];
        }
        if (mine) writeEmitter(pos, triMat, nt, sph, sphMat, i, out + 3 * (size_t)at);
        __syncthreads();
    }
    if (threadIdx.x == 0) *count = base;
}

template <class T> void upload(T *d, const std::vector<T> &v, hipStream_t stream) {
    if (!v.empty()) PT_HIP_TRY(hipMemcpyAsync(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, stream));
}

}  // namespace

void SceneArrays::load(const pt_scene &s, DevBuf &records, DevBuf &normals, float lo[3], float hi[3], hipStream_t stream) {
    nTri = (int)s.triMat.size();
    nSph = (int)s.sphMat.size();
    nMat = (int)s.mats.size();
    const int n = nTri + nSph;
    const bool smoothed = s.hasNormals && nTri > 0;
    arrays.want(pos, s.pos.size());
    arrays.want(triMat, s.triMat.size());
    arrays.want(sph, s.sph.size());
    arrays.want(sphMat, s.sphMat.size());
    arrays.want(mats, s.mats.size());
    arrays.alloc();
    WorkArrays work;
    float *nrm = nullptr, *boxes;
    uint32_t *smooth = nullptr, *rank = nullptr, *scanTmp = nullptr;
    work.want(boxes, 6 * (kBoundsBlocks + 1));
    if (smoothed) {
        work.want(nrm, s.nrm.size());
        work.want(smooth, nTri);
        work.want(rank, (size_t)nTri + 1);
        work.want(scanTmp, scanEntries(nTri));
    }
    work.alloc();
    upload(pos, s.pos, stream);
    upload(triMat, s.triMat, stream);
    upload(sph, s.sph, stream);
    upload(sphMat, s.sphMat, stream);
    upload(mats, s.mats, stream);
    if (smoothed) {
        upload(nrm, s.nrm, stream);
        k_smooth_flags<<<blocksOf(nTri), kThreads, 0, stream>>>(pos, nrm, nTri, smooth, rank);
        scanCounts(rank, nTri, scanTmp, stream);
        uint32_t kept = 0;
        PT_HIP_TRY(hipMemcpyAsync(&kept, rank + nTri, sizeof kept, hipMemcpyDeviceToHost, stream));
        PT_HIP_TRY(hipStreamSynchronize(stream));
        normals.alloc(std::max<size_t>(3 * (size_t)kept, 1) * sizeof(float4));
        k_keep_normals<<<blocksOf(nTri), kThreads, 0, stream>>>(nrm, smooth, rank, nTri, normals.as<float4>());
    } else {
        normals.alloc(sizeof(float4));
    }
    records.alloc(sizeof(float4) * 3 * (size_t)std::max(n, 1));
    k_upload_prims<<<blocksOf(n), kThreads, 0, stream>>>(pos, triMat, rank, smooth, nTri, sph, sphMat, nSph, records.as<float4>());
    const int bb = (int)std::min<unsigned>(kBoundsBlocks, blocksOf(n));
    k_bounds<<<bb, kThreads, 0, stream>>>(records.as<float4>(), n, boxes);
    k_bounds_fold<<<1, kThreads, 0, stream>>>(boxes, bb, boxes + 6 * kBoundsBlocks);
    PT_HIP_TRY(hipGetLastError());
    float b[6];
    PT_HIP_TRY(hipMemcpyAsync(b, boxes + 6 * kBoundsBlocks, sizeof b, hipMemcpyDeviceToHost, stream));
    PT_HIP_TRY(hipStreamSynchronize(stream));
    for (int k = 0; k < 3; k++) {
        lo[k] = b[k];
        hi[k] = b[3 + k];
    }
}

void SceneArrays::buildMaterials(DevBuf &records, hipStream_t stream) const {
    records.alloc(sizeof(PtMaterial) * (size_t)std::max(nMat, 1));
    if (nMat > 0) k_materials<<<blocksOf(nMat), kThreads, 0, stream>>>(mats, nMat, records.as<PtMaterial>());
    PT_HIP_TRY(hipGetLastError());
}

int SceneArrays::buildEmitters(DevBuf &records, HostInt &answer, hipStream_t stream) const {
    const int n = nTri + nSph;
    if (n <= kEmittersSmall) {
        records.alloc(sizeof(float4) * 3 * (size_t)std::max(n, 1));
        k_emitters_small<<<1, kEmittersThreads, 0, stream>>>(MaterialEdit{}, mats, nullptr, pos, triMat, nTri, sph, sphMat, nSph, 0, records.as<float4>(),
                                                             answer.target());
        PT_HIP_TRY(hipGetLastError());
        PT_HIP_TRY(hipStreamSynchronize(stream));
        return answer.read();
    }
    uint32_t count = 0, *rank, *scanTmp;
    WorkArrays work;
    work.want(rank, (size_t)n + 1);
    work.want(scanTmp, scanEntries(n));
    work.alloc();
    k_emitter_flags<<<blocksOf(n), kThreads, 0, stream>>>(mats, triMat, nTri, sphMat, nSph, rank);
    scanCounts(rank, n, scanTmp, stream);
    PT_HIP_TRY(hipMemcpyAsync(&count, rank + n, sizeof count, hipMemcpyDeviceToHost, stream));
    PT_HIP_TRY(hipStreamSynchronize(stream));
    records.alloc(sizeof(float4) * std::max<size_t>(3 * (size_t)count, 1));
    if (count > 0) {
        k_emitters<<<blocksOf(n), kThreads, 0, stream>>>(mats, pos, triMat, nTri, sph, sphMat, nSph, rank, records.as<float4>());
        PT_HIP_TRY(hipGetLastError());
        // the ranks are freed on return
        PT_HIP_TRY(hipStreamSynchronize(stream));
    }
    return (int)count;
}

int SceneArrays::editMaterial(int id, int type, const float *albedo, const float *emit, float ior, float alpha, DevBuf &materials, DevBuf &emitters,
                              int emittersNow, HostInt &answer, hipStream_t stream) {
    MaterialEdit e;
    e.id = id;
    e.setAlbedo = albedo ? 1 : 0;
    e.setEmit = emit ? 1 : 0;
    e.to.type = type;
    if (albedo) memcpy(e.to.albedo, albedo, sizeof e.to.albedo);
    if (emit) memcpy(e.to.emit, emit, sizeof e.to.emit);
    e.to.ior = ior;
    e.to.alpha = alpha;
    const bool small = nTri + nSph <= kEmittersSmall;
    if (small)
        k_emitters_small<<<1, kEmittersThreads, 0, stream>>>(e, mats, materials.as<PtMaterial>(), pos, triMat, nTri, sph, sphMat, nSph, emittersNow,
                                                             emitters.as<float4>(), answer.target());
    else k_edit_material<<<1, 64, 0, stream>>>(e, mats, materials.as<PtMaterial>(), answer.target());
    PT_HIP_TRY(hipGetLastError());
    PT_HIP_TRY(hipStreamSynchronize(stream));
    if (small) return answer.read();
    return answer.read() != 0 ? buildEmitters(emitters, answer, stream) : emittersNow;
}

// ---------------------------------------------------------------------------------------------
// Images to pageable host memory.  The runtime's own copy took 1,420 us for 24 MB and, into memory
// it had not seen, 350 us for 0.8 MB.  One copy into pinned memory takes 453 us (53 GB/s, the
// link); a piece costs 9 us more, and copying out and faulting in the destination's pages takes
// the CPU longer than the link takes, so a large image is copied out by a few threads.
// ---------------------------------------------------------------------------------------------
namespace {
constexpr size_t kReadStage = 32 << 20;     // staging memory at most
constexpr size_t kReadPieceMin = 1 << 20, kReadPieceMax = 2 << 20;
constexpr size_t kReadPerThread = 2 << 20;  // a helper thread for each such part, at most four

// Has the pages of [p, p + len) there before they are written (a new image's pages otherwise fault
// in one at a time under the copy).  Only a hint: where it fails, the copy faults them in.
void faultIn(char *p, size_t len) {
#ifdef MADV_POPULATE_WRITE
    const uintptr_t page = 4096, a = ((uintptr_t)p + page - 1) / page * page, b = ((uintptr_t)p + len) / page * page;
    if (b > a) (void)madvise((void *)a, b - a, MADV_POPULATE_WRITE);
#endif
}
}  // namespace

namespace {

// Makes a device current until it goes.
struct DeviceScope {
    int before = 0;
    bool other = false;
    explicit DeviceScope(int device) {
        PT_HIP_TRY(hipGetDevice(&before));
        other = before != device;
        if (other) PT_HIP_TRY(hipSetDevice(device));
    }
    ~DeviceScope() {
        if (other) (void)hipSetDevice(before);
    }
    DeviceScope(const DeviceScope &) = delete;
    DeviceScope &operator=(const DeviceScope &) = delete;
};

// Staging memory and its events, of one device.
struct ReadStage {
    int device = 0;
    size_t bytes = 0;
    char *p = nullptr;
    std::vector<hipEvent_t> events;
    ~ReadStage() {
        if (p) (void)hipHostFree(p);
        for (hipEvent_t e : events) (void)hipEventDestroy(e);
    }
    // false: no pinned memory to be had
    bool prepare(size_t n, size_t pieces) {
        if (bytes < n) {
            if (p) (void)hipHostFree(p);
            p = nullptr;
            bytes = 0;
            if (hipHostMalloc((void **)&p, n, hipHostMallocPortable) != hipSuccess) {
                (void)hipGetLastError();
                p = nullptr;
                return false;
            }
            bytes = n;
        }
        while (events.size() < pieces) {
            hipEvent_t e;
            PT_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            events.push_back(e);
        }
        return true;
    }
};

// One stage (at most kReadStage bytes) waits here between reads, so that a program pins memory
// once and not for every renderer it makes; reads at the same time make their own, and what is
// not taken in is freed.  Lives until the process ends.
struct StageKeeper {
    std::mutex m;
    std::unique_ptr<ReadStage> kept;
    std::unique_ptr<ReadStage> take(int device) {
        std::lock_guard<std::mutex> lock(m);
        if (kept && kept->device == device) return std::move(kept);
        auto s = std::make_unique<ReadStage>();
        s->device = device;
        return s;
    }
    void give(std::unique_ptr<ReadStage> s) {
        std::lock_guard<std::mutex> lock(m);
        if (!kept || kept->device != s->device || kept->bytes < s->bytes) std::swap(kept, s);
    }
};
StageKeeper &stageKeeper() {
    static StageKeeper *k = new StageKeeper();   // not torn down after the runtime
    return *k;
}

struct WordPage {
    static constexpr int kWords = 1024;
    std::mutex m;
    int *page = nullptr;
    std::vector<int> freed;
    int used = 0;
};
WordPage &wordPage() {
    static WordPage *w = new WordPage();
    return *w;
}

}  // namespace

HostWord::HostWord() {
    WordPage &w = wordPage();
    std::lock_guard<std::mutex> lock(w.m);
    if (!w.page && hipHostMalloc((void **)&w.page, WordPage::kWords * sizeof(int), hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        w.page = nullptr;
        return;
    }
    if (!w.freed.empty()) {
        p = w.page + w.freed.back();
        w.freed.pop_back();
    } else if (w.used < WordPage::kWords) {
        p = w.page + w.used++;
    }
    if (p) *p = 0;
}

HostWord::~HostWord() {
    if (!p) return;
    WordPage &w = wordPage();
    std::lock_guard<std::mutex> lock(w.m);
    w.freed.push_back((int)(p - w.page));
}

void readToHost(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    if (bytes == 0) return;
    // a stream takes events of its own device only, which need not be this thread's
    int device = 0;
    PT_HIP_TRY(hipStreamGetDevice(stream, &device));
    const DeviceScope on(device);
    // about six pieces
    const size_t piece = std::clamp<size_t>(bytes / 6 / 256 * 256, kReadPieceMin, kReadPieceMax);
    std::unique_ptr<ReadStage> stage = stageKeeper().take(device);
    if (!stage->prepare(std::min(bytes, kReadStage), (std::min(bytes, kReadStage) + piece - 1) / piece)) {
        PT_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream));
        PT_HIP_TRY(hipStreamSynchronize(stream));
        return;
    }
    for (size_t done = 0; done < bytes;) {
        const size_t part = std::min(bytes - done, kReadStage);
        const int n = (int)((part + piece - 1) / piece);
        char *to = (char *)dst + done, *from = stage->p;
        for (int k = 0; k < n; k++) {
            const size_t at = k * piece, len = std::min(piece, part - at);
            PT_HIP_TRY(hipMemcpyAsync(from + at, (const char *)src + done + at, len, hipMemcpyDeviceToHost, stream));
            PT_HIP_TRY(hipEventRecord(stage->events[k], stream));
        }
        std::atomic<int> next{0}, failed{0};
        auto copyOut = [&]() {
            for (int k; (k = next.fetch_add(1)) < n;) {
                const size_t at = k * piece, len = std::min(piece, part - at);
                faultIn(to + at, len);   // while the piece is on the link
                if (hipEventSynchronize(stage->events[k]) != hipSuccess) failed = 1;
                else memcpy(to + at, from + at, len);
            }
        };
        std::vector<std::thread> helpers;
        const size_t wanted = std::min<size_t>(4, part / kReadPerThread);
        try {
            while (helpers.size() < wanted) helpers.emplace_back(copyOut);
        } catch (...) {
            // no thread (or no memory for one) to be had: this one copies what is left
        }
        copyOut();
        for (std::thread &t : helpers) t.join();
        if (failed) {
            PT_HIP_TRY(hipStreamSynchronize(stream));
            throw HipFailure("waiting for an image copy failed");
        }
        done += part;
    }
    stageKeeper().give(std::move(stage));
}

}  // namespace pt
