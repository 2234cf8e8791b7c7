// pm_kernels.hip -- per-view (plain form) gfx950 kernels of the PatchMatch path.
//
// Reference behaviour (src/dense_recon/patchmatch_mvs.cu):
//   pm_init_kernel      <- init_depth_normal_kernel      (:164-216)
//   pm_cost_kernel      <- compute_ncc_cost_kernel        (:349-513)
//   pm_halfpass_kernel  <- propagate_and_refine_kernel    (:519-655)
//
// Design (gfx950, wave64):
//   * one lane per active pixel of one colour: lanes map to the compacted
//     colour lattice x = 2i + ((y + parity) & 1), so no lane idles on the
//     checkerboard;
//   * a workgroup of TX x TY lanes stages its reference window tile (with a
//     radius-wide halo, clamped at the image edge) in LDS once;
//   * per candidate and source the plane homography H = A + b (K^-T n)^T / (n.P)
//     is formed once (window centre in FP64), so a tap costs 3 FMAs for the
//     warp, one v_rcp_f32, one buffer load (the quad from the
//     row-difference plane) and 4 instructions for the bilinear sample;
//   * neighbour candidates that provably cannot win are skipped and the rest
//     shared over the workgroup's lanes (halfpass_pixel in pm_pixel.h);
//   * the five NCC moments are accumulated in FP32 on values shifted by
//     -128 DN; the variance cancellation is done in FP64.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "pm_device.h"
#include "pm_launch.h"
#include "pm_pixel.h"
#include "pm_xcd.h"

namespace hp3d {

__global__ __launch_bounds__(256) void pm_init_kernel(DevView v, uint64_t seed)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= v.W || y >= v.H) return;
    v.hyp[(x + y) & 1][y * v.Wc + (x >> 1)] = init_hyp(v, x, y, seed);
}

// Cost of the current hypotheses, run once before the first iteration: the two
// colours of a tile by neighbouring workgroups.
template <int NT, int ST, int STORE, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void pm_cost_kernel(DevView v, int tiles_x, int tiles)
{
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    __shared__ float tile[G::LH * G::LP];
    __shared__ PassXchg<TX * TY> xc;
    int t;
    if (!xcd_unit(2 * tiles, t)) return;
    const int by = (t >> 1) / tiles_x, bx = (t >> 1) - by * tiles_x;
    stage_ref_tile<R, STORE, TX, TY>(v, tile, bx, by);
    cost_tile_sorted<NT, ST, STORE, TX, TY>(v, tile, bx, by, threadIdx.x % TX, threadIdx.x / TX,
                                            t & 1, xc);
}

// Minimum waves per SIMD the half-pass's register allocation must allow.  4:
// every window's kernel fits 128 registers without spilling one (up to 40 scalar
// registers go to lanes of vector ones), and a pass issues a vector instruction
// nearly every 4 clocks; 5 would spill in the loops.
#ifndef HP3D_PLAIN_WPE
#define HP3D_PLAIN_WPE 4
#endif

// The pooled form of the refinement pays from 6 taps a row (1600x1200, 4 sources,
// FP32: 415 -> 402 us a half-pass; with 5 x 5 taps, 800x600, 3 sources, 80.7 ->
// 78.3 in means over three, but a whole solve 989 -> 1000 us over two; 3 x 3 taps,
// 1600x1200, 2 sources, 110 -> 112) and from about 3 workgroups to a CU on, where
// others fill the waits at its barriers (tiles of 32 x 8: 720x540, 816 tiles, 259
// -> 248 us with 3 sources and 11 x 11 taps; 640x480, 600 tiles, 77.2 -> 78.7 with
// 2 and 7 x 7; 480x360, 345 tiles, 66 -> 69 with 3 and 6 x 6).
constexpr int kPoolTaps = 6, kPoolTiles = 768;

template <int NT, int ST, int STORE, int TX, int TY, bool POOL>
__global__ __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(HP3D_PLAIN_WPE, 8)))
void pm_halfpass_kernel(DevView v, int iteration, int parity, uint64_t pass_seed, int tiles_x,
                        int tiles)
{
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    __shared__ float tile[G::LH * G::LP];
    __shared__ PassXchg<TX * TY> xc;
    int bx, by;
    if (!xcd_tile(tiles_x, tiles, bx, by)) return;
    stage_ref_tile<R, STORE, TX, TY>(v, tile, bx, by);
    halfpass_pixel<NT, ST, STORE, TX, TY>(v, tile, bx, by, threadIdx.x % TX, threadIdx.x / TX,
                                          iteration, parity, pass_seed, xc, POOL);
}

// Views of few pixels: up to kMaxSplitWaves waves for 64 pixels (halfpass_split).
template <int NT, int ST, int STORE, int TX, int TY>
__global__ __launch_bounds__(64 * kMaxSplitWaves)
void pm_halfpass_split_kernel(DevView v, int iteration, int parity, uint64_t pass_seed,
                              int tiles_x, int tiles)
{
    using G = TileGeom<(NT - 1) * ST / 2, STORE, TX, TY>;
    __shared__ float tile[G::LH * G::LP];
    __shared__ SplitXchg xs;
    int bx, by;
    if (!xcd_tile(tiles_x, tiles, bx, by)) return;
    halfpass_split<NT, ST, STORE, TX, TY>(v, tile, bx, by, iteration, parity, pass_seed, xs);
}

template <int NT, int ST, int STORE, int TX, int TY>
__global__ __launch_bounds__(64 * kMaxSrc)
void pm_cost_split_kernel(DevView v, int tiles_x, int tiles)
{
    using G = TileGeom<(NT - 1) * ST / 2, STORE, TX, TY>;
    __shared__ float tile[G::LH * G::LP];
    __shared__ SplitXchg xs;
    int t;
    if (!xcd_unit(2 * tiles, t)) return;
    const int by = (t >> 1) / tiles_x, bx = (t >> 1) - by * tiles_x;
    cost_split<NT, ST, STORE, TX, TY>(v, tile, bx, by, t & 1, xs);
}

// Colour planes -> row-major depth (H*W), AoS normal (H*W*3), cost and
// confidence (H*W).  Null outputs are skipped.
__global__ __launch_bounds__(256) void pm_finalize_kernel(DevView v, float* depth, float* normal,
                                                          float* cost, float* conf)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= v.W || y >= v.H) return;
    emit_pixel(v, x, y, depth, normal, cost, conf);
}

// Row-major depth + AoS normal -> colour planes (caller-given hypotheses).
__global__ __launch_bounds__(256) void pm_import_kernel(DevView v, const float* depth,
                                                        const float* normal)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= v.W || y >= v.H) return;
    const size_t q = (size_t)y * v.W + x;
    v.hyp[(x + y) & 1][y * v.Wc + (x >> 1)] =
        make_float4(depth[q], normal[3 * q], normal[3 * q + 1], normal[3 * q + 2]);
}

// 8-bit or [0,1] float gray -> the image planes (DN - 128, see pm_device.h):
// the plain plane and the row-difference gather plane
// (I[y][x], I[y+1][x] - I[y][x]), in FP32 or FP16.  in_u8 / in_f32: exactly one is non-null; in_pitch in bytes.
template <int STORE>
__global__ __launch_bounds__(256) void img_prep_kernel(const uint8_t* in_u8, const float* in_f32,
                                                       size_t in_pitch, int W, int H, void* plain,
                                                       void* coef, int pitch)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= W || y >= H) return;
    auto val = [&](int xx, int yy) -> float {
        if (in_u8) return (float)in_u8[(size_t)yy * in_pitch + xx] - kShiftDN;
        const float* row = (const float*)((const char*)in_f32 + (size_t)yy * in_pitch);
        return row[xx] * 255.0f - kShiftDN;
    };
    const float a = val(x, y);
    const size_t q = (size_t)y * pitch + x;
    // the last row's difference is never read: taps need v < H - 1
    const float dn = y < H - 1 ? val(x, y + 1) - a : 0.0f;
    if (STORE == kStoreF32) {
        static_cast<float*>(plain)[q] = a;
        static_cast<float2*>(coef)[q] = make_float2(a, dn);
    } else {
        static_cast<_Float16*>(plain)[q] = (_Float16)a;
        half2_t h;
        h.x = (_Float16)a;
        h.y = (_Float16)dn;
        static_cast<half2_t*>(coef)[q] = h;
    }
}

// One pyramid level from the previous one: element (x, y) is the mean of
// the 2 x 2 block at (2x, 2y) of the previous level's plain plane (stored
// DN - 128 values), written as the level's plain and row-difference planes.
// The sums are exact in FP32 (values carry 2 more fraction bits per level);
// FP16 storage holds the values of the first two levels and the row
// differences of the first level exactly.
template <int STORE>
__global__ __launch_bounds__(256) void img_down_kernel(const void* prev, int prev_pitch, int W,
                                                       int H, void* plain, void* coef, int pitch)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= W || y >= H) return;
    auto val = [&](int xx, int yy) -> float {
        const int q = 2 * yy * prev_pitch + 2 * xx;
        const float a = load_plain<STORE>(prev, q), b = load_plain<STORE>(prev, q + 1);
        const float c = load_plain<STORE>(prev, q + prev_pitch);
        const float d = load_plain<STORE>(prev, q + prev_pitch + 1);
        return ((a + b) + (c + d)) * 0.25f;
    };
    const size_t q = (size_t)y * pitch + x;
    if (STORE == kStoreF32) {
        const float a = val(x, y);
        const float dn = y < H - 1 ? val(x, y + 1) - a : 0.0f;
        static_cast<float*>(plain)[q] = a;
        static_cast<float2*>(coef)[q] = make_float2(a, dn);
    } else {
        // the level's stored (FP16) values, and their difference as stored
        const _Float16 a = (_Float16)val(x, y);
        const _Float16 b = (_Float16)(y < H - 1 ? val(x, y + 1) : 0.0f);
        static_cast<_Float16*>(plain)[q] = a;
        half2_t h;
        h.x = a;
        h.y = y < H - 1 ? (_Float16)((float)b - (float)a) : (_Float16)0.0f;
        static_cast<half2_t*>(coef)[q] = h;
    }
}

// ---------------------------------------------------------------------------
// Host-side launchers
// ---------------------------------------------------------------------------
static dim3 grid_2d(int W, int H) { return dim3((W + 63) / 64, (H + 3) / 4); }

hipError_t launch_init(const DevView& v, uint64_t seed, hipStream_t st)
{
    hipLaunchKernelGGL(pm_init_kernel, grid_2d(v.W, v.H), dim3(256), 0, st, v, seed);
    return hipGetLastError();
}

hipError_t launch_finalize(const DevView& v, float* depth, float* normal, float* cost, float* conf,
                           hipStream_t st)
{
    hipLaunchKernelGGL(pm_finalize_kernel, grid_2d(v.W, v.H), dim3(256), 0, st, v, depth, normal,
                       cost, conf);
    return hipGetLastError();
}

hipError_t launch_import(const DevView& v, const float* depth, const float* normal,
                         hipStream_t st)
{
    hipLaunchKernelGGL(pm_import_kernel, grid_2d(v.W, v.H), dim3(256), 0, st, v, depth, normal);
    return hipGetLastError();
}

hipError_t launch_img_prep(const uint8_t* in_u8, const float* in_f32, size_t in_pitch, int W,
                           int H, int store, void* plain, void* coef, int pitch, hipStream_t st)
{
    if (store == kStoreF32)
        hipLaunchKernelGGL(img_prep_kernel<kStoreF32>, grid_2d(W, H), dim3(256), 0, st, in_u8,
                           in_f32, in_pitch, W, H, plain, coef, pitch);
    else
        hipLaunchKernelGGL(img_prep_kernel<kStoreF16>, grid_2d(W, H), dim3(256), 0, st, in_u8,
                           in_f32, in_pitch, W, H, plain, coef, pitch);
    return hipGetLastError();
}

hipError_t launch_img_down(const void* prev, int prev_pitch, int W, int H, int store, void* plain,
                           void* coef, int pitch, hipStream_t st)
{
    if (store == kStoreF32)
        hipLaunchKernelGGL(img_down_kernel<kStoreF32>, grid_2d(W, H), dim3(256), 0, st, prev,
                           prev_pitch, W, H, plain, coef, pitch);
    else
        hipLaunchKernelGGL(img_down_kernel<kStoreF16>, grid_2d(W, H), dim3(256), 0, st, prev,
                           prev_pitch, W, H, plain, coef, pitch);
    return hipGetLastError();
}

// Workgroup tile (compacted columns x rows), from sweeps on 1600x1200 views:
// 32 x 8 (64 x 8 pixels; 32x4 and 16x16 within 1 % at 6 x 6 taps, 8x32 and
// 32x16 3 % to 15 % slower; at 11 x 11 taps 32x4, with its shorter lists, 1 to
// 2 % slower; HP3D_PLAIN_TX / _TY override both at build time).
#ifdef HP3D_PLAIN_TX
constexpr int kPlainTX = HP3D_PLAIN_TX, kPlainTY = HP3D_PLAIN_TY;
#else
constexpr int kPlainTX = 32, kPlainTY = 8;
#endif

// Whether a half-pass of `tiles` tiles takes `halves` of half the height instead:
// where the workgroups of the fullest CU then hold less of the view.  Every tile is
// in flight at once here (4 workgroups to a CU), and the launch is as long as the
// fullest CU's share: 640x480 has 600 tiles, at most 3 to a CU, against 1200 halves,
// at most 5 (half-passes of the first iteration, 2 sources, 11 x 11 taps: FP32 0.281
// ms as tiles, 0.241 as halves, FP16 0.266 and 0.237; 680x510, 704 or 1408, 3 or 6:
// 0.289 and 0.301).  In the first two iterations: later their shorter lists cost more
// (480x360, 1 source, FP32: the first two 0.029 ms faster, the next six 0.052 slower).
// Not for smaller windows, nor for 9 x 9 FP16, which gained 9 % in its first
// iteration and lost 3 % in eight.
constexpr int kCUs = 256, kHalfIterations = 2;
static bool halve_tiles(int tiles, int halves)
{
    return (halves + kCUs - 1) / kCUs < 2 * ((tiles + kCUs - 1) / kCUs);
}

// The split kernels' tile: 16 x 4 (32 x 4 pixels; 32x2 and 8x8 within 3 %).
constexpr int kSplitTX = 16, kSplitTY = 4;

// Waves of a split workgroup for a view of n such tiles, 0: not split.  Split,
// every wave repeats the pixel's bookkeeping and the rounds are not pooled, so
// it pays only while the plain kernel's n / 4 workgroups leave SIMDs idle for
// the length of their chain of S sources: up to n = 400 S for windows of up to
// 49 taps, 750 S above.  Half-pass, plain -> split, at and beyond the line:
//   6x6 taps: 480x360 S=8 0.161 -> 0.123 ms, 560x420 S=4 0.092 -> 0.093,
//             641x479 S=5 0.139 -> 0.143, 800x600 S=8 0.268 -> 0.283
//   11x11:    480x360 S=2 0.135 -> 0.120, 560x420 S=2 0.140 -> 0.151,
//             800x600 S=6 0.617 -> 0.604, 1280x960 S=5 1.217 -> 1.254
// 4 waves a workgroup fill a CU best (S = 5 with 6: a CU holds 2 such
// workgroups, 12 of its 16 waves; +20 %); the smallest views, whose waves do
// not fill the chip at 8 a workgroup either, are fastest with 8, and with room
// for both refinement steps (3 S) below 160 tiles.  96x72, S=8, 6x6 taps:
// 0.138 ms plain, 0.054 with 4 waves, 0.039 with 8, 0.036 with 16.
static int split_waves(int NT, int n, int S)
{
    if (n > (NT * NT >= 81 ? 750 : 400) * S) return 0;
    return n > 300 ? 4 : n > 160 ? 8 : std::min(kMaxSplitWaves, std::max(8, 3 * S));
}

// The same for the initial cost, whose workgroups have no chain but the
// sources: up to n = 1600 S (800x600, S=6, 11x11: 0.400 -> 0.322 ms for both
// colours, 1280x960 S=8 1.18 -> 1.05, S=3 at 6x6 0.153 -> 0.154, 1600x1200 S=4
// 0.286 -> 0.320).
static int cost_split_waves(int n, int S)
{
    if (n > 1600 * S || S < 2) return 0;
    return std::min(n > 300 ? 4 : 8, S);
}

template <int NT, int ST, int STORE>
static void launch_pass_t(const DevView& v, int mode, int iteration, int parity,
                          uint64_t pass_seed, hipStream_t st)
{
    const int sx = (v.Wc + kSplitTX - 1) / kSplitTX, sn = sx * ((v.H + kSplitTY - 1) / kSplitTY);
    const int waves = mode == kPassCost ? cost_split_waves(sn, v.S) : split_waves(NT, sn, v.S);
    if (waves && mode == kPassCost) {
        hipLaunchKernelGGL((pm_cost_split_kernel<NT, ST, STORE, kSplitTX, kSplitTY>),
                           dim3(xcd_grid(2 * sn)), dim3(64 * waves), 0, st, v, sx, sn);
        return;
    }
    if (waves) {
        hipLaunchKernelGGL((pm_halfpass_split_kernel<NT, ST, STORE, kSplitTX, kSplitTY>),
                           dim3(xcd_grid(sn)), dim3(64 * waves), 0, st, v, iteration, parity,
                           pass_seed, sx, sn);
        return;
    }
    constexpr int kTX = kPlainTX, kTY = kPlainTY;
    const int tiles_x = (v.Wc + kTX - 1) / kTX;
    const int tiles = tiles_x * ((v.H + kTY - 1) / kTY);
    constexpr bool kHalf = (NT >= 11 || (NT >= 9 && STORE == kStoreF32)) && kTX * kTY % 128 == 0;
    constexpr int kHalfTY = kHalf ? kTY / 2 : kTY;
    const int halves = tiles_x * ((v.H + kHalfTY - 1) / kHalfTY);
    if (mode == kPassCost)
        hipLaunchKernelGGL((pm_cost_kernel<NT, ST, STORE, kTX, kTY>), dim3(xcd_grid(2 * tiles)),
                           dim3(kTX * kTY), 0, st, v, tiles_x, tiles);
    else if (NT >= kPoolTaps && tiles >= kPoolTiles && pool_refinement(v.S, v.top_k, iteration))
        hipLaunchKernelGGL((pm_halfpass_kernel<NT, ST, STORE, kTX, kTY, (NT >= kPoolTaps)>),
                           dim3(xcd_grid(tiles)), dim3(kTX * kTY), 0, st, v, iteration, parity,
                           pass_seed, tiles_x, tiles);
    else if (kHalf && tiles < kPoolTiles && iteration < v.first_iteration + kHalfIterations &&
             halve_tiles(tiles, halves))
        hipLaunchKernelGGL((pm_halfpass_kernel<NT, ST, STORE, kTX, kHalfTY, false>),
                           dim3(xcd_grid(halves)), dim3(kTX * kHalfTY), 0, st, v, iteration, parity,
                           pass_seed, tiles_x, halves);
    else
        hipLaunchKernelGGL((pm_halfpass_kernel<NT, ST, STORE, kTX, kTY, false>),
                           dim3(xcd_grid(tiles)), dim3(kTX * kTY), 0, st, v, iteration, parity,
                           pass_seed, tiles_x, tiles);
}

template <int STORE>
static bool dispatch_window(const DevView& v, int radius, int stride, int mode, int iteration,
                            int parity, uint64_t pass_seed, hipStream_t st)
{
#define HP3D_CASE(R_, S_)                                                                   \
    if (radius == R_ && stride == S_) {                                                     \
        launch_pass_t<(2 * R_) / S_ + 1, S_, STORE>(v, mode, iteration, parity, pass_seed, st); \
        return true;                                                                        \
    }
    HP3D_CASE(1, 1) HP3D_CASE(2, 1) HP3D_CASE(3, 1) HP3D_CASE(4, 1) HP3D_CASE(5, 1)
    HP3D_CASE(1, 2) HP3D_CASE(2, 2) HP3D_CASE(3, 2) HP3D_CASE(4, 2) HP3D_CASE(5, 2)
#undef HP3D_CASE
    return false;
}

bool window_supported(int radius, int stride)
{
    return radius >= 1 && radius <= 5 && (stride == 1 || stride == 2);
}

hipError_t launch_pass(const DevView& v, int store, int radius, int stride, int mode,
                       int iteration, int parity, uint64_t pass_seed, hipStream_t st)
{
    const bool ok = store == kStoreF32
                        ? dispatch_window<kStoreF32>(v, radius, stride, mode, iteration, parity,
                                                     pass_seed, st)
                        : dispatch_window<kStoreF16>(v, radius, stride, mode, iteration, parity,
                                                     pass_seed, st);
    if (!ok) return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace hp3d
