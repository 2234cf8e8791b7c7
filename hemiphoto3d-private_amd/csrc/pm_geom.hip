// pm_geom.hip -- geometric consistency filter over a set of depth maps.
//
// Reference: geometric_consistency_filter_kernel (src/dense_recon/
// patchmatch_mvs.cu:668-781) and its driver (:1267-1384).  The driver walks
// the views in order; view i is filtered against its sources' depth maps as
// they are at that moment, so a source earlier in the order contributes its
// already-filtered map.  Here every map is uploaded once and stays on the
// device; one launch per view in the same order reproduces that dependence,
// and the single-precision operations are written in the reference's order
// (this file is compiled without contraction), so the result is bit-exact
// with an FP32 restatement of the same loop.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "pm_runtime.h"
#include "pm_xcd.h"

namespace hp3d {

struct GeomSrcDev {
    float K[9], R[9], t[3];
    const float* depth;
    const float* normal;
};

struct GeomViewDev {
    float kinv[9], R[9], t[3];
    int W, H, S, min_consistent;
    float tol, cos_tol;
    float* depth;
    const float* normal;
    float* conf;
    GeomSrcDev src[kMaxSrc];
};

// Whether pixel (x, y) of depth d > 0 (or NaN) is seen at its depth by enough
// sources.
__device__ __forceinline__ bool geom_consistent(const GeomViewDev& g, int x, int y, size_t idx,
                                                float d)
{
    const float* ki = g.kinv;
    const float* R = g.R;
    const float fx = (float)x, fy = (float)y;
    // back-project, then to world: P_w = R^T (P_c - t)
    const float pcx = d * (ki[0] * fx + ki[1] * fy + ki[2]);
    const float pcy = d * (ki[3] * fx + ki[4] * fy + ki[5]);
    const float pcz = d * (ki[6] * fx + ki[7] * fy + ki[8]);
    const float a = pcx - g.t[0], b = pcy - g.t[1], c = pcz - g.t[2];
    const float pwx = R[0] * a + R[3] * b + R[6] * c;
    const float pwy = R[1] * a + R[4] * b + R[7] * c;
    const float pwz = R[2] * a + R[5] * b + R[8] * c;
    const float ncx = g.normal[3 * idx], ncy = g.normal[3 * idx + 1], ncz = g.normal[3 * idx + 2];
    const float nwx = R[0] * ncx + R[3] * ncy + R[6] * ncz;
    const float nwy = R[1] * ncx + R[4] * ncy + R[7] * ncz;
    const float nwz = R[2] * ncx + R[5] * ncy + R[8] * ncz;
    int consistent = 0;
    for (int s = 0; s < g.S; ++s) {
        const GeomSrcDev& sv = g.src[s];
        const float psx = sv.R[0] * pwx + sv.R[1] * pwy + sv.R[2] * pwz + sv.t[0];
        const float psy = sv.R[3] * pwx + sv.R[4] * pwy + sv.R[5] * pwz + sv.t[1];
        const float psz = sv.R[6] * pwx + sv.R[7] * pwy + sv.R[8] * pwz + sv.t[2];
        if (psz <= 0.0f) continue;
        const float prx = sv.K[0] * psx + sv.K[1] * psy + sv.K[2] * psz;
        const float pry = sv.K[3] * psx + sv.K[4] * psy + sv.K[5] * psz;
        const float prz = sv.K[6] * psx + sv.K[7] * psy + sv.K[8] * psz;
        const float u = prx / prz, w = pry / prz;
        const float ru = rintf(u), rw = rintf(w);   // round to nearest even (__float2int_rn)
        // bounds tested in float first: values beyond int range are out anyway
        if (!(ru >= 0.0f && ru < (float)g.W && rw >= 0.0f && rw < (float)g.H)) continue;
        const size_t sp = (size_t)(int)rw * g.W + (int)ru;
        const float ds = sv.depth[sp];
        if (ds <= 0.0f) continue;
        if (fabsf(ds - psz) / psz > g.tol) continue;
        const float nsx = sv.normal[3 * sp], nsy = sv.normal[3 * sp + 1], nsz = sv.normal[3 * sp + 2];
        const float swx = sv.R[0] * nsx + sv.R[3] * nsy + sv.R[6] * nsz;
        const float swy = sv.R[1] * nsx + sv.R[4] * nsy + sv.R[7] * nsz;
        const float swz = sv.R[2] * nsx + sv.R[5] * nsy + sv.R[8] * nsz;
        if (nwx * swx + nwy * swy + nwz * swz < g.cos_tol) continue;
        consistent++;
    }
    return consistent >= g.min_consistent;
}

// One 64x4-pixel tile per workgroup, tiles in XCD order: the source maps'
// rows that a band of the view projects to stay in one XCD's L2.  Bound by its
// gathers (44 us for a 1280x960 view with 8 sources, 3.6 TB/s).  kept[tile]:
// pixels left with a depth, which a pass over the downloaded maps on the host
// took 1.1 ms to count for nine such views (null: not counted).
__global__ __launch_bounds__(256) void geom_filter_kernel(GeomViewDev g, int tiles_x, int tiles,
                                                          int* kept)
{
    int bx, by;
    if (!xcd_tile(tiles_x, tiles, bx, by)) return;
    const int x = bx * 64 + (threadIdx.x & 63);
    const int y = by * 4 + (threadIdx.x >> 6);
    bool left = false;
    if (x < g.W && y < g.H) {
        const size_t idx = (size_t)y * g.W + x;
        const float d = g.depth[idx];
        if (d <= 0.0f) {
            if (g.conf) g.conf[idx] = 0.0f;
        } else if (geom_consistent(g, x, y, idx, d)) {
            left = d > 0.0f;
        } else {
            g.depth[idx] = 0.0f;
            if (g.conf) g.conf[idx] = 0.0f;
        }
    }
    const int n = __syncthreads_count(left);
    if (kept && threadIdx.x == 0) kept[by * tiles_x + bx] = n;
}

}  // namespace hp3d

using namespace hp3d;

extern "C" int hp3d_pm_geom_filter(hp3d_pm_ctx* ctx, hp3d_geom_view* views, int n,
                                   float depth_tol, float normal_tol_deg, int min_consistent,
                                   int* retained)
{
    if (!ctx) return HP3D_ERR_INVALID_ARG;
    if (!views || n < 1 || min_consistent < 0 || !(depth_tol >= 0.0f))
        return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: bad arguments");
    for (int i = 0; i < n; ++i) {
        const hp3d_geom_view& v = views[i];
        if (v.width < 1 || v.height < 1 || !v.depth || !v.normal || v.num_src < 0 ||
            v.num_src > kMaxSrc)
            return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: view %d is malformed", i);
        // a view's own map is filtered in place while its sources are read,
        // so it must not be one of them; a repeated source would count twice
        for (int s = 0; s < v.num_src; ++s) {
            if (v.src[s] < 0 || v.src[s] >= n)
                return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: view %d source %d out of range", i, s);
            if (v.src[s] == i)
                return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: view %d lists itself as a source", i);
            for (int r = 0; r < s; ++r)
                if (v.src[r] == v.src[s])
                    return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: view %d lists source %d twice",
                                     i, v.src[s]);
        }
    }
    (void)hipSetDevice(ctx->device);
    // one device block: per view depth, normal, confidence
    std::vector<size_t> off(n);
    size_t total = 0;
    for (int i = 0; i < n; ++i) {
        off[i] = total;
        const size_t px = (size_t)views[i].width * views[i].height;
        total += ((px * 5 * sizeof(float)) + 255) & ~(size_t)255;
    }
    // and the tiles' counts of pixels left
    auto tiles_of = [&](int i) { return ((views[i].width + 63) / 64) * ((views[i].height + 3) / 4); };
    std::vector<size_t> tile_base(n + 1, 0);
    for (int i = 0; i < n; ++i) tile_base[i + 1] = tile_base[i] + tiles_of(i);
    void* block = nullptr;
    const size_t maps = total;
    total += tile_base[n] * sizeof(int);
    int rc = ctx->dev_alloc(&block, total, "geometric filter maps");
    if (rc) {   // maps that just fit: counted on the host
        total = maps;
        rc = ctx->dev_alloc(&block, total, "geometric filter maps");
    }
    if (rc) return rc;
    auto dptr = [&](int i, int k) {   // k: 0 depth, 1 normal, 4 confidence
        const size_t px = (size_t)views[i].width * views[i].height;
        return reinterpret_cast<float*>(static_cast<char*>(block) + off[i]) + (k == 4 ? 4 * px : k * px);
    };
    std::vector<HostLink::Seg> segs;
    for (int i = 0; i < n; ++i) {
        const size_t px = (size_t)views[i].width * views[i].height * 4;
        segs.push_back({views[i].depth, dptr(i, 0), px});
        segs.push_back({const_cast<float*>(views[i].normal), dptr(i, 1), 3 * px});
        if (views[i].confidence) segs.push_back({views[i].confidence, dptr(i, 4), px});
    }
    hipError_t e = ctx->link.upload(segs, ctx->stream);
    int* const d_kept =
        total > maps ? reinterpret_cast<int*>(static_cast<char*>(block) + maps) : nullptr;
    const float cos_tol = std::cos(normal_tol_deg * 3.14159265358979323846f / 180.0f);
    std::vector<char> filtered(n, 0);
    double ki[9];
    for (int i = 0; i < n && e == hipSuccess; ++i) {
        const hp3d_geom_view& v = views[i];
        GeomViewDev g;
        std::memset(&g, 0, sizeof g);
        // sources with a different size are skipped (:1310)
        for (int s = 0; s < v.num_src; ++s) {
            const hp3d_geom_view& sv = views[v.src[s]];
            if (sv.width != v.width || sv.height != v.height) continue;
            GeomSrcDev& d = g.src[g.S++];
            for (int k = 0; k < 9; ++k) { d.K[k] = (float)sv.K[k]; d.R[k] = (float)sv.R[k]; }
            for (int k = 0; k < 3; ++k) d.t[k] = (float)sv.t[k];
            d.depth = dptr(v.src[s], 0);
            d.normal = dptr(v.src[s], 1);
        }
        if (g.S < min_consistent) continue;   // view left unfiltered (:1330)
        if (hp3d_pm_invert3(v.K, ki) != HP3D_OK) {
            (void)ctx->dev_free(block, total);
            return ctx->fail(HP3D_ERR_INVALID_ARG, "geom_filter: view %d K is singular", i);
        }
        for (int k = 0; k < 9; ++k) { g.kinv[k] = (float)ki[k]; g.R[k] = (float)v.R[k]; }
        for (int k = 0; k < 3; ++k) g.t[k] = (float)v.t[k];
        g.W = v.width;
        g.H = v.height;
        g.min_consistent = min_consistent;
        g.tol = depth_tol;
        g.cos_tol = cos_tol;
        g.depth = dptr(i, 0);
        g.normal = dptr(i, 1);
        g.conf = v.confidence ? dptr(i, 4) : nullptr;
        const int tiles_x = (v.width + 63) / 64, tiles = tiles_of(i);
        hipLaunchKernelGGL(geom_filter_kernel, dim3(xcd_grid(tiles)), dim3(256), 0, ctx->stream, g,
                           tiles_x, tiles, d_kept ? d_kept + tile_base[i] : nullptr);
        e = hipGetLastError();
        filtered[i] = 1;
    }
    segs.clear();
    for (int i = 0; i < n; ++i) {
        const size_t px = (size_t)views[i].width * views[i].height * 4;
        segs.push_back({views[i].depth, dptr(i, 0), px});
        if (views[i].confidence) segs.push_back({views[i].confidence, dptr(i, 4), px});
    }
    // (the kernel's counts are each view's own; where views share host memory, the
    // bytes that stay are the later one's and are counted there)
    std::vector<int> kept(retained && d_kept && !HostLink::overlap(segs.data(), segs.size()) ? tile_base[n] : 0);
    if (!kept.empty()) segs.push_back({kept.data(), d_kept, kept.size() * sizeof(int)});
    if (e == hipSuccess) e = ctx->link.download(segs, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    ctx->dev_free(block, total);
    if (e != hipSuccess) return ctx->hip_fail(e, "geometric filter");
    if (retained)
        for (int i = 0; i < n; ++i) {
            int r = 0;
            if (!kept.empty()) {
                for (size_t t = tile_base[i]; t < tile_base[i + 1] && filtered[i]; ++t) r += kept[t];
            } else {
                const size_t px = (size_t)views[i].width * views[i].height;
                for (size_t p = 0; p < px; ++p) r += views[i].depth[p] > 0.0f;
            }
            retained[i] = filtered[i] ? r : -1;
        }
    return HP3D_OK;
}
