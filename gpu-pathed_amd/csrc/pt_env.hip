// pt_env.hip -- environment importance-sampling tables built on the GPU in FP64.
//
// Weight of texel (x, y) = r + g + b (environment_light.cu:44-47), optionally times
// sin(theta).  Every row and the marginal over the row sums get an alias table by the sweep
// construction (heavy items absorb the deficits of light items in index order; a heavy item
// whose residual drops below one becomes a light bucket aliased to the next heavy item).  The
// operation order is fixed and fused multiply-adds are disabled here, so the tables are
// reproducible bit for bit.
//
// The sums and the sweeps are serial chains of FP64 additions whose order is part of the
// result; what bounds the build is the latency of one link times the row length (bytes and
// operations would take 7 us on a 1024x512 map).  One wave per row: the wave loads, weighs and
// sorts the row's texels into light and heavy ones 64 at a time, and only the chain itself runs
// on wave-uniform values, fed from lane registers (v_readlane); which item a step settled is
// worked out afterwards, a step per lane.  The marginal table is block 0 of the same launch: it
// needs the row sums only.  On that map: weights and sums 14 us, sweeps 68 us (50 ns a step; 117
// us with a branch per step, 146 us with the branches nested), densities 5 us; one thread per
// row over global memory and the marginal after it took 2,650 us in all.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/pathed.h"
#include "pt_gpu.h"
#include "pt_internal.h"

#pragma clang fp contract(off)

namespace pt {

namespace {

// Texel weights and their row's sum, in index order.  One wave per row: kSumTile weights at a
// time go to LDS and are added as broadcast reads, which keeps the chain at the latency of one
// FP64 addition.
constexpr int kSumTile = 512;
__device__ __forceinline__ double chainSum(const double *tile, int n, double sum) {
    int k = 0;
    for (; k + 16 <= n; k += 16) {
        double v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = tile[k + q];
#pragma unroll
        for (int q = 0; q < 16; q++) sum += v[q];
    }
    for (; k < n; k++) sum += tile[k];
    return sum;
}
__global__ __launch_bounds__(64) void k_env_weights(const float4 *rgba, int w, int h, int sinWeight, double *wts, double *rowSum) {
    __shared__ double tile[kSumTile];
    const int y = blockIdx.x, lane = threadIdx.x;
    const double st = sinWeight ? sin((y + 0.5) / h * 3.14159265358979323846) : 1.0;
    const float4 *src = rgba + (size_t)y * w;
    double *dst = wts + (size_t)y * w;
    double sum = 0.0;
    for (int x0 = 0; x0 < w; x0 += kSumTile) {
        const int n = min(kSumTile, w - x0);
#pragma unroll
        for (int k = 0; k < kSumTile; k += 64) {
            const int x = k + lane;
            if (x < n) {
                const float4 v = src[x0 + x];
                const double wt = ((double)v.x + (double)v.y + (double)v.z) * st;
                dst[x0 + x] = wt;
                tile[x] = wt;
            }
        }
        __syncthreads();
        sum = chainSum(tile, n, sum);
        __syncthreads();
    }
    if (lane == 0) rowSum[y] = sum;
}

// Sweep steps between two looks at the item lists.
constexpr int kSweepSteps = 24;

// 64 items of a list around the sweep's position in it, one per lane, and the 64 items from
// that position on, already loading.  A window is used for kSweepSteps steps from where the
// last ones ended and then replaced: at most 2 kSweepSteps + 1 of its items are looked at.
struct SweepWindow {
    const int *list;       // item indices and their scaled weights; entries `step` apart
    const double *scaled;
    int step;              // +1 (light items, from the front) or -1 (heavy items, from the back)
    int count;             // items of the list
    double past;           // the weight that stands behind the last item
    int pos;               // list position of the sweep
    int at;                // the window lane of that position
    int idx, nextIdx;
    double q, nextQ;

    __device__ __forceinline__ void prefetch() {
        const int k = pos + (int)threadIdx.x;
        // the list has an item where it is read at all (a lane past its end reads the last)
        const int64_t o = (int64_t)step * min(k, count - 1);
        if (count > 0) {
            nextIdx = list[o];
            nextQ = scaled[o];
        }
    }
    __device__ __forceinline__ void take(int first) {
        idx = nextIdx;
        q = first + (int)threadIdx.x < count ? nextQ : past;
    }
    __device__ __forceinline__ void start() {
        pos = 0;
        at = 0;
        nextIdx = 0;
        nextQ = 0.0;
        prefetch();
        take(0);
        prefetch();
    }
    // the position has moved to window lane `to`
    __device__ __forceinline__ void advance(int to) {
        const int first = pos;     // where the window that is already loading starts
        pos += to - at;
        at = to - at;
        take(first);
        prefetch();
    }
};

__device__ __forceinline__ double laneDouble(double v, int lane) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// The alias table of w[0 .. n) (sum: their sum in index order) by one wave: table entries
// (probability as float, alias as int bits) and, with WIDE, the FP64 probabilities and
// aliases.  list, scaled: n entries each of working memory.
template <bool WIDE>
__device__ __forceinline__ void aliasSweep(const double *w, int n, double sum, int *list, double *scaled, float2 *table, double *probOut, int *aliasOut) {
    const int lane = threadIdx.x;
    auto put = [&](int i, double prob, int alias) {
        table[i] = make_float2((float)prob, asFloat(alias));
        if constexpr (WIDE) {
            probOut[i] = prob;
            aliasOut[i] = alias;
        }
    };
    const bool some = sum > 0.0;
    const double scale = (double)n / sum;
    // light items (scaled weight below one) to the front of the list, heavy ones to its back
    int nLight = 0, nHeavy = 0;
    const uint64_t below = lane == 0 ? 0ull : ~0ull >> (64 - lane);
    for (int x0 = 0; x0 < n; x0 += 256) {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = w[min(x0 + 64 * k + lane, n - 1)];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int x = x0 + 64 * k + lane;
            const bool in = x < n;
            const double q = v[k] * scale;
            const bool light = in && some && q < 1.0;
            const uint64_t mL = __ballot(light), mH = __ballot(in && !light);
            const int o = light ? nLight + __popcll(mL & below) : n - 1 - (nHeavy + __popcll(mH & below));
            if (in) {
                list[o] = x;
                scaled[o] = q;
            }
            nLight += __popcll(mL);
            nHeavy += __popcll(mH);
        }
    }
    if (!some || nHeavy == 0) {
        for (int x = lane; x < n; x += 64) put(x, 1.0, x);
        return;
    }
    // the wave reads what its other lanes stored
    __threadfence_block();
    // A light item behind the last one takes nothing and a heavy one behind the last leaves
    // nothing: the sweep then steps past the end of that list until the batch is over.
    SweepWindow L{list, scaled, 1, nLight, 1.0}, H{list + (n - 1), scaled + (n - 1), -1, nHeavy, -INFINITY};
    L.start();
    H.start();
    double wj = laneDouble(H.q, 0);   // what is left of the heavy item at H.pos
    // every step moves one of the positions on, so the loop ends after at most n + 1 steps
    while (L.pos <= nLight && H.pos < nHeavy) {
        // The chain, without branches: one step is a comparison and both candidates for the next
        // residual (a branch taken costs a single wave more than they do).  Lane s keeps the
        // residual that step s found.
        const double d = L.q - 1.0;
        double found = 0.0;
        int li = L.at;
        const int ends = L.at + H.at + 1;   // one step moves one of the two
#pragma unroll
        for (int s = 0; s < kSweepSteps; s++) {
            found = lane == s ? wj : found;
            const bool ge = wj >= 1.0;
            const double filled = wj + laneDouble(d, li), passed = laneDouble(H.q, ends + s - li) + (wj - 1.0);
            wj = ge ? filled : passed;
            li += (int)(__ballot(ge) & 1);
        }
        const int hi = ends - 1 + kSweepSteps - li;
        // lane s settles step s: a light item filled by the current heavy one, or the residual
        // heavy item as a light bucket of the next
        const bool fill = found >= 1.0;
        const uint64_t m = __ballot(fill && lane < kSweepSteps);
        const int fills = __popcll(m & below);
        const int l = L.at + fills, h = H.at + (min(lane, kSweepSteps) - fills);
        const int light = __shfl(L.idx, l), cur = __shfl(H.idx, h), next = __shfl(H.idx, h + 1);
        const double lightQ = __shfl(L.q, l);
        if (lane < kSweepSteps) {
            if (fill) {
                if (L.pos + fills < nLight) put(light, lightQ, cur);
            } else if (H.pos + (lane - fills) + 1 < nHeavy) {
                put(cur, found, next);
            }
        }
        L.advance(li);
        H.advance(hi);
    }
    // items that the sweep did not reach keep probability one: the light ones left and the
    // heavy ones from the one being emptied on
    for (int k = L.pos + lane; k < nLight; k += 64) put(list[k], 1.0, list[k]);
    for (int k = min(H.pos, nHeavy - 1) + lane; k < nHeavy; k += 64) put(list[n - 1 - k], 1.0, list[n - 1 - k]);
}

// The FP64 working arrays of one table build; the FP64 tables are all there or all null.
struct EnvScratch {
    double *wts, *rowSum, *total, *rowScaled, *margScaled;
    int *rowList, *margList;
    double *rowProb, *margProb;
    int *rowAlias, *margAlias;
};

// Block 0: the marginal table and the total; block 1 + y: row y's table.
template <bool WIDE>
__global__ __launch_bounds__(64) void k_env_sweeps(EnvScratch s, int w, int h, float2 *rows, float2 *marginal) {
    if (blockIdx.x > 0) {
        const int y = (int)blockIdx.x - 1;
        const size_t o = (size_t)y * w;
        aliasSweep<WIDE>(s.wts + o, w, s.rowSum[y], s.rowList + o, s.rowScaled + o, rows + o, s.rowProb + o, s.rowAlias + o);
        return;
    }
    __shared__ double tile[kSumTile];
    double sum = 0.0;
    for (int y0 = 0; y0 < h; y0 += kSumTile) {
        const int n = min(kSumTile, h - y0);
        for (int k = threadIdx.x; k < n; k += 64) tile[k] = s.rowSum[y0 + k];
        __syncthreads();
        sum = chainSum(tile, n, sum);
        __syncthreads();
    }
    if (threadIdx.x == 0) *s.total = sum;
    aliasSweep<WIDE>(s.rowSum, h, sum, s.margList, s.margScaled, marginal, s.margProb, s.margAlias);
}

__global__ void k_env_pdf(const double *wts, const double *total, int w, int h, float *texelPdf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w * h) return;
    const double t = *total;
    const double norm = t > 0.0 ? (double)w * h / (2.0 * 3.14159265358979323846 * 3.14159265358979323846) / t : 0.0;
    texelPdf[i] = (float)(wts[i] * norm);
}

}  // namespace

__global__ void k_env_pack_pdf(float4 *rgba, const float *texelPdf, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) rgba[i].w = texelPdf[i];
}

void packEnvPdf(float4 *rgba, const float *texelPdf, int n, hipStream_t stream) {
    if (n <= 0) return;
    k_env_pack_pdf<<<(n + 255) / 256, 256, 0, stream>>>(rgba, texelPdf, n);
    PT_HIP_TRY(hipGetLastError());
}

namespace {

void launchEnvTables(const float4 *rgba, int w, int h, int sinWeight, const EnvScratch &s, float2 *rows, float2 *marginal,
                     float *texelPdf, hipStream_t stream) {
    const size_t n = (size_t)w * h;
    k_env_weights<<<h, 64, 0, stream>>>(rgba, w, h, sinWeight, s.wts, s.rowSum);
    if (s.rowProb) k_env_sweeps<true><<<h + 1, 64, 0, stream>>>(s, w, h, rows, marginal);
    else k_env_sweeps<false><<<h + 1, 64, 0, stream>>>(s, w, h, rows, marginal);
    k_env_pdf<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(s.wts, s.total, w, h, texelPdf);
    PT_HIP_TRY(hipGetLastError());
}

}  // namespace

void buildEnvTables(const float4 *rgba, int w, int h, int sinWeight, float2 *rows, float2 *marginal, float *texelPdf, double *rowProbOut,
                    int *rowAliasOut, double *margProbOut, int *margAliasOut, hipStream_t stream) {
    const size_t n = (size_t)w * h;
    DevBuf wts, rs, tot, rl, ml, rq, mq, rp, ra, mp, ma;
    wts.alloc(n * sizeof(double));
    rs.alloc(h * sizeof(double));
    tot.alloc(sizeof(double));
    rl.alloc(n * sizeof(int));
    ml.alloc(h * sizeof(int));
    rq.alloc(n * sizeof(double));
    mq.alloc(h * sizeof(double));
    if (rowProbOut || rowAliasOut || margProbOut || margAliasOut) {
        rp.alloc(n * sizeof(double));
        ra.alloc(n * sizeof(int));
        mp.alloc(h * sizeof(double));
        ma.alloc(h * sizeof(int));
    }
    const EnvScratch sc{wts.as<double>(), rs.as<double>(), tot.as<double>(), rq.as<double>(), mq.as<double>(), rl.as<int>(), ml.as<int>(),
                        rp.as<double>(), mp.as<double>(), ra.as<int>(), ma.as<int>()};
    launchEnvTables(rgba, w, h, sinWeight, sc, rows, marginal, texelPdf, stream);
    if (rowProbOut) PT_HIP_TRY(hipMemcpyAsync(rowProbOut, rp.p, n * sizeof(double), hipMemcpyDeviceToHost, stream));
    if (rowAliasOut) PT_HIP_TRY(hipMemcpyAsync(rowAliasOut, ra.p, n * sizeof(int), hipMemcpyDeviceToHost, stream));
    if (margProbOut) PT_HIP_TRY(hipMemcpyAsync(margProbOut, mp.p, h * sizeof(double), hipMemcpyDeviceToHost, stream));
    if (margAliasOut) PT_HIP_TRY(hipMemcpyAsync(margAliasOut, ma.p, h * sizeof(int), hipMemcpyDeviceToHost, stream));
    // temporaries are freed on return: wait for the kernels that read them
    PT_HIP_TRY(hipStreamSynchronize(stream));
}

// ---------------------------------------------------------------------------------------------
// Table build without allocation: the working arrays live in one fixed device array per GPU.
// ---------------------------------------------------------------------------------------------
namespace {

constexpr size_t kAlign = 256;
constexpr size_t alignUp(size_t b) { return (b + kAlign - 1) / kAlign * kAlign; }
constexpr size_t scratchBytes(size_t texels, size_t rows) {
    return alignUp(texels * sizeof(double)) * 2 + alignUp(texels * sizeof(int)) + alignUp(rows * sizeof(double)) * 2 +
           alignUp(rows * sizeof(int)) + alignUp(sizeof(double));
}
constexpr size_t kScratchBytes = scratchBytes(PT_ENV_NOALLOC_MAX_TEXELS, PT_ENV_NOALLOC_MAX_ROWS);

// Device-side working memory of pt_env_tables_noalloc.  Host code never uses this name as an
// address (on the host it is a stand-in symbol): it uses the per-device pointer that
// hipGetSymbolAddress returns.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex gScratchMutex;
void *gScratchPtr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device.
void *scratchOnDevice(int dev) {
    std::lock_guard<std::mutex> lock(gScratchMutex);
    if (!gScratchPtr[dev]) {
        void *ptr = nullptr;
        PT_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) throw HipFailure("hipGetSymbolAddress(scratch) returned NULL");
        gScratchPtr[dev] = ptr;
    }
    return gScratchPtr[dev];
}

}  // namespace

}  // namespace pt

extern "C" int pt_env_tables_noalloc(const float *rgba, int width, int height, int sin_theta_weight, float *rows, float *marginal,
                                     float *texel_pdf, void *stream) {
    using namespace pt;
    if (!rgba || !rows || !marginal || !texel_pdf || width <= 0 || height <= 0)
        return fail(PT_ERR_INVALID, "pt_env_tables_noalloc: bad arguments");
    if ((int64_t)width * height > PT_ENV_NOALLOC_MAX_TEXELS || height > PT_ENV_NOALLOC_MAX_ROWS)
        return fail(PT_ERR_INVALID, "pt_env_tables_noalloc: map of " + std::to_string(width) + "x" + std::to_string(height) +
                                        " exceeds the fixed scratch (at most " + std::to_string(PT_ENV_NOALLOC_MAX_TEXELS) +
                                        " texels and " + std::to_string(PT_ENV_NOALLOC_MAX_ROWS) + " rows)");
    try {
        int dev = 0;
        PT_HIP_TRY(hipGetDevice(&dev));
        if (dev < 0 || dev >= kMaxDevices) return fail(PT_ERR_DEVICE, "pt_env_tables_noalloc: device ordinal out of range");
        unsigned char *base = (unsigned char *)scratchOnDevice(dev);
        const size_t n = (size_t)width * height, hh = (size_t)height;
        EnvScratch sc{};   // without the FP64 tables
        size_t at = 0;
        auto carve = [&](size_t bytes) {
            unsigned char *p = base + at;
            at += alignUp(bytes);
            return p;
        };
        sc.wts = (double *)carve(n * sizeof(double));
        sc.rowScaled = (double *)carve(n * sizeof(double));
        sc.rowList = (int *)carve(n * sizeof(int));
        sc.rowSum = (double *)carve(hh * sizeof(double));
        sc.margScaled = (double *)carve(hh * sizeof(double));
        sc.margList = (int *)carve(hh * sizeof(int));
        sc.total = (double *)carve(sizeof(double));
        if (at > kScratchBytes) return fail(PT_ERR_INVALID, "pt_env_tables_noalloc: scratch layout exceeds its array");
        // every working array is written in full before it is read, so nothing is cleared
        launchEnvTables((const float4 *)rgba, width, height, sin_theta_weight, sc, (float2 *)rows, (float2 *)marginal, texel_pdf,
                        (hipStream_t)stream);
        return PT_OK;
    } catch (const HipFailure &e) {
        return fail(PT_ERR_DEVICE, std::string("pt_env_tables_noalloc: ") + e.msg);
    }
}
