// pm_fuse.hip -- depth-map fusion into a point cloud.
//
// Reference: fuseDepthMaps (src/dense_recon/point_cloud.h:7-9) is declared
// as the consumer of the MVS depth and normal maps but is a stub returning an
// empty cloud (point_cloud.cu:4-8).  This is the natural device form of it:
// every pixel with depth > 0 (and confidence >= min_confidence when a
// confidence map is given) becomes one point, in view order then row-major
// pixel order:
//   position = R^T (d K^-1 [x, y, 1] - t)   (world frame, include/types.h:55-74)
//   normal   = R^T n                        (camera -> world)
//   colour   = the pixel's 8-bit value / 255 (gray replicated, or RGB)
// A count pass over every view, one scan of the per-block counts and a write
// pass place every point at its row-major rank, so the output is
// deterministic; each pass is one launch over all views.  The maps come over
// the link, which bounds the whole call: a call that only counts uploads depth
// and confidence.  Single-precision operations are written in one fixed order
// (no contraction), which the oracle restates.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "pm_runtime.h"

namespace hp3d {

namespace {

constexpr int kFuseBlock = 256;
// Pixels of a workgroup, kFuseBlock at a time: an eighth of the counts to scan
// (five 1280x960 views: count and scan 5 x 15 us in ten launches of 256-pixel
// blocks, one launch each now).
constexpr int kFuseSpan = 8 * kFuseBlock;

struct FuseViewDev {
    float kinv[9], R[9], t[3];
    int W, H, channels;
    float min_conf;
    const float* depth;
    const float* normal;
    const float* conf;
    const uint8_t* color;
    int first_block;   // of the launch's blocks, in view order
};

__device__ __forceinline__ bool fuse_valid(const FuseViewDev& g, int q)
{
    const float d = g.depth[q];
    return d > 0.0f && (!g.conf || g.conf[q] >= g.min_conf);
}

// The view of this block: the last with first_block <= blockIdx.x.
__device__ __forceinline__ const FuseViewDev& fuse_view(const FuseViewDev* views, int n)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (views[mid].first_block <= (int)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    return views[lo];
}

__global__ __launch_bounds__(kFuseBlock) void fuse_count_kernel(const FuseViewDev* views, int n,
                                                                int* counts)
{
    const FuseViewDev& g = fuse_view(views, n);
    const long long q0 = (long long)((int)blockIdx.x - g.first_block) * kFuseSpan + threadIdx.x;
    const long long px = (long long)g.W * g.H;
    __shared__ int part[kFuseBlock / 64];
    int c = 0;
#pragma unroll
    for (int k = 0; k < kFuseSpan; k += kFuseBlock)
        c += __popcll(__ballot(q0 + k < px && fuse_valid(g, (int)(q0 + k))));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int w = 0; w < kFuseBlock / 64; ++w) s += part[w];
        counts[blockIdx.x] = s;
    }
}

// Exclusive scan of n block counts from `base` on (one workgroup; n is at most a few
// hundred thousand), its end into *total.
__global__ __launch_bounds__(1024) void fuse_scan_kernel(const int* counts, int n, long long base,
                                                         long long* offsets, long long* total)
{
    __shared__ long long carry;
    __shared__ long long part[1024 / 64];
    if (threadIdx.x == 0) carry = base;
    __syncthreads();
    for (int start = 0; start < n; start += 1024) {
        const int i = start + threadIdx.x;
        const long long c = i < n ? counts[i] : 0;
        // inclusive scan within the wave
        long long x = c;
        const int lane = threadIdx.x & 63;
        for (int o = 1; o < 64; o <<= 1) {
            const long long y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) part[threadIdx.x >> 6] = x;
        __syncthreads();
        if (threadIdx.x == 0) {
            long long s = 0;
            for (int w = 0; w < 1024 / 64; ++w) {
                const long long p = part[w];
                part[w] = s;
                s += p;
            }
        }
        __syncthreads();
        if (i < n) offsets[i] = carry + part[threadIdx.x >> 6] + x - c;
        __syncthreads();
        if (threadIdx.x == 1023) carry = carry + part[15] + x;
        __syncthreads();
    }
    if (threadIdx.x == 0) *total = carry;
}

// The point of pixel q, written at rank o.
__device__ __forceinline__ void fuse_point(const FuseViewDev& g, int q, long long o, float* pos,
                                           float* nrm, float* col)
{
    const int y = q / g.W, x = q - y * g.W;
    const float d = g.depth[q];
    const float fx = (float)x, fy = (float)y;
    const float* ki = g.kinv;
    const float* R = g.R;
    const float pcx = d * (ki[0] * fx + ki[1] * fy + ki[2]);
    const float pcy = d * (ki[3] * fx + ki[4] * fy + ki[5]);
    const float pcz = d * (ki[6] * fx + ki[7] * fy + ki[8]);
    const float a = pcx - g.t[0], b = pcy - g.t[1], c = pcz - g.t[2];
    pos[3 * o] = R[0] * a + R[3] * b + R[6] * c;
    pos[3 * o + 1] = R[1] * a + R[4] * b + R[7] * c;
    pos[3 * o + 2] = R[2] * a + R[5] * b + R[8] * c;
    if (nrm) {
        float nx = 0.0f, ny = 0.0f, nz = 0.0f;
        if (g.normal) {
            nx = g.normal[3 * (size_t)q];
            ny = g.normal[3 * (size_t)q + 1];
            nz = g.normal[3 * (size_t)q + 2];
        }
        nrm[3 * o] = R[0] * nx + R[3] * ny + R[6] * nz;
        nrm[3 * o + 1] = R[1] * nx + R[4] * ny + R[7] * nz;
        nrm[3 * o + 2] = R[2] * nx + R[5] * ny + R[8] * nz;
    }
    if (col) {
        float r = 0.0f, gg = 0.0f, bb = 0.0f;
        if (g.color && g.channels == 1) {
            r = gg = bb = (float)g.color[q] / 255.0f;
        } else if (g.color && g.channels == 3) {
            r = (float)g.color[3 * (size_t)q] / 255.0f;
            gg = (float)g.color[3 * (size_t)q + 1] / 255.0f;
            bb = (float)g.color[3 * (size_t)q + 2] / 255.0f;
        }
        col[3 * o] = r;
        col[3 * o + 1] = gg;
        col[3 * o + 2] = bb;
    }
}

__global__ __launch_bounds__(kFuseBlock) void fuse_write_kernel(const FuseViewDev* views, int n,
                                                                const long long* offsets,
                                                                float* pos, float* nrm, float* col)
{
    const FuseViewDev& g = fuse_view(views, n);
    const long long q0 = (long long)((int)blockIdx.x - g.first_block) * kFuseSpan + threadIdx.x;
    const long long px = (long long)g.W * g.H;
    __shared__ int part[2][kFuseBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    long long base = offsets[blockIdx.x];
    for (int k = 0; k < kFuseSpan / kFuseBlock; ++k) {
        const long long q = q0 + k * kFuseBlock;
        const bool v = q < px && fuse_valid(g, (int)q);
        const unsigned long long m = __ballot(v);
        // (two sets: the next row's counts are written while this one's are read)
        if (lane == 0) part[k & 1][wave] = __popcll(m);
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < kFuseBlock / 64; ++w) {
            if (w < wave) before += part[k & 1][w];
            all += part[k & 1][w];
        }
        if (v)
            fuse_point(g, (int)q, base + before + __popcll(m & ((1ull << lane) - 1ull)), pos, nrm,
                       col);
        base += all;
    }
}

size_t a256(size_t b) { return (b + 255) & ~(size_t)255; }
size_t fuse_blocks(size_t px) { return (px + kFuseSpan - 1) / kFuseSpan; }

// One attempt at hp3d_pm_fuse, its arguments checked.  All views at once, or
// (one_by_one) count, scan and write view after view, which takes less memory for
// the view table, counts and offsets.  *refused: the memory was not to be had.
int fuse_views(hp3d_pm_ctx* ctx, const hp3d_fuse_view* views, int n, float min_confidence,
               float* positions, float* normals, float* colors, size_t capacity, size_t* count,
               bool one_by_one, bool* refused)
{
    *refused = false;
    // what the call needs on the device: to count, depth and confidence; to
    // write, the maps of what it writes.  One device block: the maps, then the total,
    // the views, offsets and counts.
    const bool write = positions != nullptr;
    std::vector<FuseViewDev> g(n);
    std::vector<HostLink::Seg> segs;   // device: offsets into the block, for now
    size_t total = 0, blocks = 0, largest = 0;
    auto put = [&](const void* host, size_t bytes) {
        const size_t off = total;
        segs.push_back({const_cast<void*>(host), reinterpret_cast<void*>(off), bytes});
        total += a256(bytes);
        return off;
    };
    struct Offsets { size_t depth, normal, conf, color; };
    std::vector<Offsets> off(n);
    for (int i = 0; i < n; ++i) {
        const hp3d_fuse_view& v = views[i];
        const size_t px = (size_t)v.width * v.height;
        FuseViewDev& d = g[i];
        std::memset(&d, 0, sizeof d);
        double ki[9];
        if (hp3d_pm_invert3(v.K, ki) != HP3D_OK)
            return ctx->fail(HP3D_ERR_INVALID_ARG, "fuse: view %d K is singular", i);
        for (int k = 0; k < 9; ++k) { d.kinv[k] = (float)ki[k]; d.R[k] = (float)v.R[k]; }
        for (int k = 0; k < 3; ++k) d.t[k] = (float)v.t[k];
        d.W = v.width;
        d.H = v.height;
        d.channels = v.color ? v.color_channels : 0;
        d.min_conf = min_confidence;
        d.first_block = one_by_one ? 0 : (int)blocks;
        off[i].depth = put(v.depth, px * 4);
        if (v.confidence) off[i].conf = put(v.confidence, px * 4);
        if (write && normals && v.normal) off[i].normal = put(v.normal, px * 12);
        if (write && colors && v.color) off[i].color = put(v.color, px * v.color_channels);
        blocks += fuse_blocks(px);
        largest = std::max(largest, fuse_blocks(px));
    }
    // (view by view, less than a total, offsets and counts of 256-pixel blocks take)
    const size_t held = one_by_one ? 1 : n, rows = one_by_one ? largest : blocks;
    const size_t scratch = total;
    const size_t offsets_off = scratch + 8 + held * sizeof(FuseViewDev);
    static_assert(sizeof(FuseViewDev) % 8 == 0, "offsets aligned after the views");
    total += a256(8 + held * sizeof(FuseViewDev) + rows * 12);
    void* block = nullptr;
    int rc = ctx->dev_alloc(&block, total, "fusion maps");
    if (rc) {
        *refused = true;
        return rc;
    }
    char* base = static_cast<char*>(block);
    long long* d_total = reinterpret_cast<long long*>(base + scratch);
    FuseViewDev* d_views = reinterpret_cast<FuseViewDev*>(base + scratch + 8);
    long long* d_offsets = reinterpret_cast<long long*>(base + offsets_off);
    int* d_counts = reinterpret_cast<int*>(base + offsets_off + rows * 8);
    for (auto& s : segs) s.dev = base + reinterpret_cast<size_t>(s.dev);
    for (int i = 0; i < n; ++i) {
        const hp3d_fuse_view& v = views[i];
        g[i].depth = reinterpret_cast<const float*>(base + off[i].depth);
        if (v.confidence) g[i].conf = reinterpret_cast<const float*>(base + off[i].conf);
        if (write && normals && v.normal) g[i].normal = reinterpret_cast<const float*>(base + off[i].normal);
        if (write && colors && v.color) g[i].color = reinterpret_cast<const uint8_t*>(base + off[i].color);
    }
    if (!one_by_one) segs.push_back({g.data(), d_views, n * sizeof(FuseViewDev)});
    hipError_t e = ctx->link.upload(segs, ctx->stream);
    // the views of group k, their blocks, and the ranks of their points from `from` on
    const int groups = one_by_one ? n : 1, group_views = one_by_one ? 1 : n;
    auto group_blocks = [&](int k) {
        return one_by_one ? fuse_blocks((size_t)g[k].W * g[k].H) : blocks;
    };
    auto rank = [&](int k, long long from) -> hipError_t {
        if (one_by_one) {
            const hipError_t ue = ctx->link.upload({{&g[k], d_views, sizeof(FuseViewDev)}}, ctx->stream);
            if (ue != hipSuccess) return ue;
        }
        hipLaunchKernelGGL(fuse_count_kernel, dim3((unsigned)group_blocks(k)), dim3(kFuseBlock), 0,
                           ctx->stream, d_views, group_views, d_counts);
        hipLaunchKernelGGL(fuse_scan_kernel, dim3(1), dim3(1024), 0, ctx->stream, d_counts,
                           (int)group_blocks(k), from, d_offsets, d_total);
        return hipGetLastError();
    };
    std::vector<long long> from(groups + 1, 0);
    for (int k = 0; k < groups && e == hipSuccess; ++k) {
        e = rank(k, from[k]);
        if (e == hipSuccess) e = ctx->link.download({{&from[k + 1], d_total, sizeof(long long)}}, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    }
    if (e != hipSuccess) {
        ctx->dev_free(block, total);
        return ctx->hip_fail(e, "fusion count");
    }
    const size_t npts = (size_t)from[groups];
    *count = npts;
    if (!positions || npts == 0) {
        ctx->dev_free(block, total);
        return HP3D_OK;
    }
    if (capacity < npts) {
        ctx->dev_free(block, total);
        return ctx->fail(HP3D_ERR_INVALID_ARG, "fuse: %zu points exceed the capacity %zu", npts,
                         capacity);
    }
    // write into one device output block, then copy out
    void* out = nullptr;
    const size_t per = npts * 12;
    const int nbuf = 1 + (normals ? 1 : 0) + (colors ? 1 : 0);
    rc = ctx->dev_alloc(&out, per * nbuf, "fusion output");
    if (rc) {
        ctx->dev_free(block, total);
        *refused = true;
        return rc;
    }
    float* d_pos = static_cast<float*>(out);
    float* d_nrm = normals ? d_pos + 3 * npts : nullptr;
    float* d_col = colors ? d_pos + 3 * npts * (normals ? 2 : 1) : nullptr;
    for (int k = 0; k < groups && e == hipSuccess; ++k) {
        if (one_by_one) e = rank(k, from[k]);
        if (e != hipSuccess) break;
        hipLaunchKernelGGL(fuse_write_kernel, dim3((unsigned)group_blocks(k)), dim3(kFuseBlock), 0,
                           ctx->stream, d_views, group_views, d_offsets, d_pos, d_nrm, d_col);
        e = hipGetLastError();
    }
    segs.assign({{positions, d_pos, per}});
    if (normals) segs.push_back({normals, d_nrm, per});
    if (colors) segs.push_back({colors, d_col, per});
    if (e == hipSuccess) e = ctx->link.download(segs, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    ctx->dev_free(out, per * nbuf);
    ctx->dev_free(block, total);
    if (e != hipSuccess) return ctx->hip_fail(e, "fusion");
    return HP3D_OK;
}

}  // namespace

}  // namespace hp3d

using namespace hp3d;

extern "C" int hp3d_pm_fuse(hp3d_pm_ctx* ctx, const hp3d_fuse_view* views, int n,
                            float min_confidence, float* positions, float* normals,
                            float* colors, size_t capacity, size_t* count)
{
    if (!ctx) return HP3D_ERR_INVALID_ARG;
    if (!views || n < 1 || !count || !(min_confidence == min_confidence))
        return ctx->fail(HP3D_ERR_INVALID_ARG, "fuse: bad arguments");
    size_t blocks = 0;
    for (int i = 0; i < n; ++i) {
        const hp3d_fuse_view& v = views[i];
        if (v.width < 1 || v.height < 1 || !v.depth ||
            (long long)v.width * v.height > (1ll << 31) - kFuseBlock ||
            (v.color && v.color_channels != 1 && v.color_channels != 3))
            return ctx->fail(HP3D_ERR_INVALID_ARG, "fuse: view %d is malformed", i);
        blocks += fuse_blocks((size_t)v.width * v.height);
    }
    (void)hipSetDevice(ctx->device);
    // all views at once, unless a launch cannot hold them (2^32 threads) or their
    // table and counts are what does not fit
    bool refused = blocks >= 0xffffffffull / kFuseBlock;
    int rc = HP3D_OK;
    if (!refused)
        rc = fuse_views(ctx, views, n, min_confidence, positions, normals, colors, capacity, count,
                        false, &refused);
    if (refused)
        rc = fuse_views(ctx, views, n, min_confidence, positions, normals, colors, capacity, count,
                        true, &refused);
    return rc;
}
