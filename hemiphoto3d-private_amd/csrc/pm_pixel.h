// pm_pixel.h -- per-pixel device functions of the PatchMatch path, shared by
// the per-view kernels (pm_kernels.hip) and the multi-view step kernel
// (pm_step.hip).  Every function here is a pure function of its arguments and
// the view's state, so a pixel computes the same bits in either kernel.
//
// Reference behaviour (src/dense_recon/patchmatch_mvs.cu):
//   init_hyp        <- init_depth_normal_kernel      (:164-216)
//   cand_cost       <- computePixelCost               (:222-343)
//   cost_pixel      <- compute_ncc_cost_kernel body   (:349-513)
//   halfpass_pixel  <- propagate_and_refine_kernel    (:519-655)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pm_device.h"
#include "pm_window.h"

// Build-time choice of the half-pass's depth-ordered candidate list: the
// number of leading iterations of a solve that order a wave's candidates by
// depth (1, the default: the first; 0: owner order in every iteration).
#ifndef HP3D_BUCKET
#define HP3D_BUCKET 1
#endif
// Build-time choice of the windows (by tap count) whose tap coordinates are
// taken relative to an integer base near the window centre's source position
// (default: up to 5x5 taps, the windows whose NCC a sub-pixel coordinate
// error moves the most; 0: none; taken to every window it measured 1.5-4 %
// slower at 36 and 121 taps, for no gain in accuracy there).
#ifndef HP3D_LOCAL_TAPS
#define HP3D_LOCAL_TAPS 25
#endif
// Build-time choice of the windows (by tap count) whose taps run from the
// centre on (centre row, the rows below it, then the rows above; the same for
// the columns of a row), so that the window's first tap is its centre; the
// others run top-left first.  Default: from 7x7 taps up, where the moment
// sums' rounding needed it; below, the centre-first order measured slower
// (its gathers hit the L1 cache less) for no gain in accuracy.
#ifndef HP3D_CENTRE_FIRST_TAPS
#define HP3D_CENTRE_FIRST_TAPS 49
#endif

namespace hp3d {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Philox4x32-10 and the u01 mapping ((x >> 8) + 1) * 2^-24 in (0, 1].
// ---------------------------------------------------------------------------
__device__ __forceinline__ void philox(uint32_t& c0, uint32_t& c1, uint32_t& c2, uint32_t& c3,
                                       uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) { k0 += kPhiloxW0; k1 += kPhiloxW1; }
        const uint32_t hi0 = __umulhi(kPhiloxM0, c0), lo0 = kPhiloxM0 * c0;
        const uint32_t hi1 = __umulhi(kPhiloxM1, c2), lo1 = kPhiloxM1 * c2;
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    }
}

__device__ __forceinline__ float u01(uint32_t x)
{
    return (float)((x >> 8) + 1u) * (1.0f / 16777216.0f);
}

// Unit view ray K^-1 [x, y, 1] / |.|, written so it rounds like the host code.
__device__ __forceinline__ void unit_ray(const float* ki, int x, int y, float& rx, float& ry,
                                         float& rz)
{
    const float fx = (float)x, fy = (float)y;
    float a = ki[0] * fx + ki[1] * fy + ki[2];
    float b = ki[3] * fx + ki[4] * fy + ki[5];
    float c = ki[6] * fx + ki[7] * fy + ki[8];
    const float len = sqrtf(a * a + b * b + c * c);
    if (len > 1e-12f) { a = a / len; b = b / len; c = c / len; }
    rx = a; ry = b; rz = c;
}

// Unnormalised ray K^-1 [x, y, 1] in FP64 (the cost's back-projection, :241-243).
__device__ __forceinline__ void ray_fp64(const double* ki, int x, int y, double& rx, double& ry,
                                         double& rz)
{
    const double X = x, Y = y;
    rx = ki[0] * X + ki[1] * Y + ki[2];
    ry = ki[3] * X + ki[4] * Y + ki[5];
    rz = ki[6] * X + ki[7] * Y + ki[8];
}

// ---------------------------------------------------------------------------
// Image element access
// ---------------------------------------------------------------------------
template <int STORE> __device__ __forceinline__ float load_plain(const void* p, int off);
template <> __device__ __forceinline__ float load_plain<kStoreF32>(const void* p, int off)
{
    return static_cast<const float*>(p)[off];
}
template <> __device__ __forceinline__ float load_plain<kStoreF16>(const void* p, int off)
{
    return (float)static_cast<const _Float16*>(p)[off];
}

// Planes are read through buffer resources: the hardware range-checks every
// access and returns 0 outside the plane, so a tap whose computed address is
// wild (a lane that will be masked) can never fault.  Dword 3 = 0x00020000 is
// the raw 32-bit data format of gfx9-family buffer descriptors.
//   stride 0 (raw): num_records counts bytes and the load takes a byte
//     offset, checked against it;
//   stride s (structured, the source gather planes): num_records counts
//     records of s bytes and the load takes a record index, which the buffer
//     unit checks against num_records and scales by s.  The check is on the
//     index alone: a 16-byte load at an 8-byte stride returns the record and
//     its successor in full (measured on gfx950).
constexpr int kBufferRsrcWord3 = 0x00020000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int num_records, short stride = 0)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), stride, num_records, kBufferRsrcWord3);
}

typedef int v4i32_t __attribute__((ext_vector_type(4)));
typedef int v2i32_t __attribute__((ext_vector_type(2)));
// Structured buffer loads (the LLVM intrinsics; hipcc has no builtin for them).
__device__ v4i32_t struct_load_b128(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                    int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v4i32");
__device__ v2i32_t struct_load_b64(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                   int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v2i32");
// A record index past every gather plane (a plane holds at most
// kMaxPlaneBytes, so fewer records): the load is range-checked away and
// returns zeros.
constexpr unsigned kIdxNowhere = 0x7ffffff0u;
static_assert(kIdxNowhere >= kMaxPlaneBytes, "index inside a plane");

// Access to the hypothesis state planes (hyp, cost, change flags).
// COH = false: ordinary loads and stores (one kernel launch per pass: the
// launch boundary orders passes).  COH = true: device-coherent accesses
// (the sc1 cache policy, bypassing the per-CU L1 and the per-XCD L2 caches
// that are not coherent across XCDs), for the persistent batch kernel, where
// a tile's pass reads what workgroups on other XCDs wrote in the same launch.
// The image planes are read-only within a launch and keep ordinary cached
// loads either way.  Planes addressed this way hold less than 2 GiB.
// How the persistent kernel keeps the state planes coherent across XCDs
// (build-time choice, measured): bit 0 set = its state stores are ordinary
// stores followed by an agent-scope release fence (an L2 write-back) before a
// tile's counter moves, else device-coherent (sc1) stores; bit 1 set = its
// state loads are ordinary loads after an agent-scope acquire fence (an L2
// invalidate) once the tile's dependencies are met, else sc1 loads.
#ifndef HP3D_PERSIST_MEM
#define HP3D_PERSIST_MEM 0
#endif
constexpr bool kPersistPlainStores = (HP3D_PERSIST_MEM & 1) != 0;
constexpr bool kPersistPlainLoads = (HP3D_PERSIST_MEM & 2) != 0;

template <bool COH> struct StateIO;
template <> struct StateIO<false> {
    static __device__ __forceinline__ float4 ld4(const float4* p, int i) { return p[i]; }
    static __device__ __forceinline__ float ld1(const float* p, int i) { return p[i]; }
    static __device__ __forceinline__ unsigned ldb(const unsigned char* p, int i) { return p[i]; }
    static __device__ __forceinline__ void st4(float4* p, int i, float4 x) { p[i] = x; }
    static __device__ __forceinline__ void st1(float* p, int i, float x) { p[i] = x; }
    static __device__ __forceinline__ void stb(unsigned char* p, int i, unsigned x)
    {
        p[i] = (unsigned char)x;
    }
};
template <> struct StateIO<true> {
    static constexpr int kSC1 = 16;   // cache-policy operand: sc1 (device scope)
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rs(const void* p)
    {
        return make_rsrc(p, 0x7fffffff);
    }
    static constexpr int kLd = kPersistPlainLoads ? 0 : kSC1;
    static constexpr int kSt = kPersistPlainStores ? 0 : kSC1;
    static __device__ __forceinline__ float4 ld4(const float4* p, int i)
    {
        return __builtin_bit_cast(float4,
                                  __builtin_amdgcn_raw_buffer_load_b128(rs(p), i * 16, 0, kLd));
    }
    static __device__ __forceinline__ float ld1(const float* p, int i)
    {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs(p), i * 4, 0, kLd));
    }
    static __device__ __forceinline__ unsigned ldb(const unsigned char* p, int i)
    {
        return __builtin_amdgcn_raw_buffer_load_b8(rs(p), i, 0, kLd);
    }
    static __device__ __forceinline__ void st4(float4* p, int i, float4 x)
    {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, x),
                                               rs(p), i * 16, 0, kSt);
    }
    static __device__ __forceinline__ void st1(float* p, int i, float x)
    {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), rs(p), i * 4, 0, kSt);
    }
    static __device__ __forceinline__ void stb(unsigned char* p, int i, unsigned x)
    {
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)x, rs(p), i, 0, kSt);
    }
};

// Bilinear sample at (ix + au, iy + aw) of the texel quad a = I[iy][ix],
// b = I[iy][ix+1], c = I[iy+1][ix], d = I[iy+1][ix+1].  Both storages keep a
// row-difference plane for source gathers, element (x, y) =
// (I[y][x], I[y+1][x] - I[y][x]), so that one load per tap at (ix, iy)
// returns the whole quad as (a, c - a, b, d - b): 16 bytes from 8 bytes per
// pixel (F32) or 8 bytes from 4 (F16).  The sample is then two FMAs down the
// columns and a subtract and an FMA across -- 4 VALU instructions, against 6
// for three lerps of a row-pair plane (a, c, b, d) -- in FP32 either way.
// For 8-bit images the values (DN - 128) and the row differences (at most
// 255 in magnitude) are integers, exact in FP16, so both storages give
// identical results.  (Measured on 1600x1200 views: one load per tap instead
// of one per texel row, 1.6x at stride 2; the F16 plane's halved footprint
// 1.13x more at stride 1; differences instead of row pairs, +2 % (F32) /
// +5 % (F16) at stride 2 and +16 % at stride 1.)
// A source's gather plane as records of one texel (FP32: 8 bytes, FP16: 4):
// the load takes the record index iy * pitch + ix (one multiply-add per tap)
// and reads that texel's record and its right neighbour's, (a, c-a, b, d-b).
// A valid tap has ix <= W-2 and iy <= H-2, so both records lie inside the
// plane; an invalid tap's index goes nowhere and reads zeros.
template <int STORE> struct SrcImage;
template <> struct SrcImage<kStoreF32> {
    typedef float4 Quad;
    __amdgpu_buffer_rsrc_t rsrc;
    unsigned pitch;
    __device__ SrcImage(const DevView& v, int s)
        : rsrc(make_rsrc(v.src_coef[s], v.coef_bytes / 8, 8)), pitch((unsigned)v.pitch_plain) {}
    __device__ __forceinline__ unsigned index(int ix, int iy, bool ok) const
    {
        const unsigned idx = __umul24((unsigned)iy, pitch) + (unsigned)ix;
        return ok ? idx : kIdxNowhere;
    }
    __device__ __forceinline__ Quad load(unsigned idx) const
    {
        return __builtin_bit_cast(float4, struct_load_b128(rsrc, (int)idx, 0, 0, 0));
    }
    static __device__ __forceinline__ float lerp(const Quad& q, float au, float aw)
    {
        const float c0 = fmaf(aw, q.y, q.x), c1 = fmaf(aw, q.w, q.z);
        return fmaf(au, c1 - c0, c0);
    }
};
template <> struct SrcImage<kStoreF16> {
    typedef half4_t Quad;
    __amdgpu_buffer_rsrc_t rsrc;
    unsigned pitch;
    __device__ SrcImage(const DevView& v, int s)
        : rsrc(make_rsrc(v.src_coef[s], v.coef_bytes / 4, 4)), pitch((unsigned)v.pitch_plain) {}
    __device__ __forceinline__ unsigned index(int ix, int iy, bool ok) const
    {
        const unsigned idx = __umul24((unsigned)iy, pitch) + (unsigned)ix;
        return ok ? idx : kIdxNowhere;
    }
    __device__ __forceinline__ Quad load(unsigned idx) const
    {
        return __builtin_bit_cast(half4_t, struct_load_b64(rsrc, (int)idx, 0, 0, 0));
    }
    static __device__ __forceinline__ float lerp(const Quad& q, float au, float aw)
    {
        const float c0 = fmaf(aw, (float)q.y, (float)q.x), c1 = fmaf(aw, (float)q.w, (float)q.z);
        return fmaf(au, c1 - c0, c0);
    }
};

// floor(x) converted to int in one instruction (v_cvt_flr_i32_f32; out of
// range saturates, which the unsigned bounds test then rejects).
__device__ __forceinline__ int cvt_flr(float x)
{
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

struct TapSums {
    float sr, ss, srr, sss, srs;
    int cnt;
};

// Sums of the reference window over every tap, in tap order: they do not
// depend on the candidate or the source, so a window whose taps are all
// valid takes them from here instead of accumulating them per source.
struct WinRef {
    float sr, srr;
};
template <int NT, int ST>
__device__ __forceinline__ WinRef window_ref_sums(const float* __restrict__ lwin, int lp)
{
    constexpr int F = NT * NT >= HP3D_CENTRE_FIRST_TAPS ? NT / 2 : 0;   // first row and column
    float sr = 0.f, srr = 0.f;
#pragma unroll 1
    for (int jr = 0; jr < NT; ++jr) {
        const int j = jr + F < NT ? jr + F : jr + F - NT;
        const float* lrow = lwin + j * ST * lp;
#pragma unroll
        for (int ir = 0; ir < NT; ++ir) {
            const int i = ir + F < NT ? ir + F : ir + F - NT;
            const float r = lrow[i * ST];
            sr += r;
            srr = fmaf(r, r, srr);
        }
    }
    return WinRef{sr, srr};
}

// Taps of a window row whose gathers are in flight together (C of tap_window).
// Half-pass: rows of up to 7 taps whole, 9 and 11 taps as 5 + 4 and 6 + 5.  With
// two whole rows of 11 in flight (as many gathers as the compiler would keep
// registers for) that kernel held 167 registers and 3 waves to a SIMD, its
// unrolled loops filled more than the 64 KiB instruction cache, and a change
// anywhere else could make it wait for each gather by itself (+23 % time); in
// chunks it holds 123 (FP16 111), 4 waves, and every loop is one row long: 1280x960
// with 8 sources at stride 1, FP32, 2.00 -> 1.94 ms a half-pass.
// Initial cost: whole rows.  Its random hypotheses scatter the gathers, the
// L1's line rate bounds it, and chunks only add to its waits (1600x1200, 4 sources,
// 11x11 taps, FP32: 0.86 against 0.92 ms).
template <int NT> constexpr int kPassChunk = NT <= 7 ? NT : (NT + 1) / 2;
template <int NT> constexpr int kCostChunk = NT;
constexpr int kOutsideTaps = 4;   // taps a row from which source_cost tests window_outside

// The window's taps for one candidate and source (patchmatch_mvs.cu:273-307).
// MASKED = false is used only when every tap is known to be inside the image;
// it takes the reference sums from wr, which window_ref_sums forms with the
// same additions in the same order as the masked loop does when every tap is
// valid, so a window's sums do not depend on which variant its wave ran.
//
// The source moments are taken of s - s0, with s0 the window's first valid
// sample (the NCC is invariant to a constant shift of the samples).  Unshifted,
// a low-contrast window's samples sit far from zero (up to 128 DN against a
// spread of a few DN), and the FP32 rounding of s^2 and of the running sums
// carries over into n*sum(s^2) - sum(s)^2 amplified by mean^2 / variance: up
// to 1.2e-3 of cost error on small views.  Shifted, the summands are of the
// size of the spread.  When every tap is valid both loops take the first
// tap's sample, so the variants still agree bit for bit.  In windows of 7x7
// taps and more the taps run from the window centre on (window_ref_sums in
// the same order), so s0 is the centre's sample: near the window mean, the
// running sums of s - s0 wander instead of growing with the tap count, and
// sum(r (s - s0)), whose reference values are not shifted, rounds 3-4x less
// over 121 taps.
//
// (cx, cy) and the columns (h00, h10), (h01, h11) may be relative to an
// integer base (bu, bv): the taps' coordinates are then u - bu and v - bv,
// and the base is added back to the texel index.
//
// A row's neighbouring taps read the same cache lines, 64 a gather where the
// hypotheses are random, and the L1 holds four gathers' worth: the row's gathers
// have to come back to back, before other waves' push those lines out.  In the
// initial cost the compiler does that by itself, but in the masked loop of 11 FP32
// quads it put 13 instructions of address arithmetic between any two.  BURST forms
// all addresses first: 11 x 11 taps, 2400x1800, 6 sources, 3.80 -> 3.01 ms (with 3
// waves to a SIMD instead of 4, 3.49 and 3.01); 3200x2400, 3 sources, 3.30 -> 2.79;
// 1600x1200, 4 sources, 0.93 -> 0.86.  (The persistent kernel's START, with 3 waves
// and nothing sorted, lost 8 % by it.)
template <int NT, int ST, int STORE, bool MASKED, bool ZCHK, int C, bool BURST>
__device__ __forceinline__ void tap_window(const SrcImage<STORE>& img,
                                           const float* __restrict__ lwin, int lp, float cx,
                                           float cy, float cz, float h00, float h01, float h10,
                                           float h11, float h20, float h21, unsigned umax,
                                           unsigned vmax, const WinRef& wr, TapSums& m,
                                           int bu = 0, int bv = 0)
{
    constexpr int R = (NT - 1) * ST / 2;
    constexpr int F = NT * NT >= HP3D_CENTRE_FIRST_TAPS ? NT / 2 : 0;   // first row and column
    float sr = 0.f, ss = 0.f, srr = 0.f, sss = 0.f, srs = 0.f;
    float s0 = 0.f;     // the shift: first valid sample of the window
    bool have = false;  // (masked loop) a valid tap has been seen
    int cnt = 0;
#pragma unroll 1
    for (int jr = 0; jr < NT; ++jr) {
        const int j = jr + F < NT ? jr + F : jr + F - NT;
        const float oy = (float)(j * ST - R);
        const float bx = fmaf(h01, oy, cx);
        const float by = fmaf(h11, oy, cy);
        const float bz = fmaf(h21, oy, cz);
        const float* lrow = lwin + j * ST * lp;
#pragma unroll
        for (int i0 = 0; i0 < NT; i0 += C) {
            constexpr bool kBurst = MASKED && BURST;
            static_assert(!kBurst || C == NT, "whole rows");
            typename SrcImage<STORE>::Quad q[C];
            unsigned idx[C];
            float au[C], aw[C], rv[C];
            bool okv[C];
#pragma unroll
            for (int t = 0; t < C; ++t) {
                const int ir = i0 + t;
                if (ir >= NT) break;
                const int i = ir + F < NT ? ir + F : ir + F - NT;
                const float ox = (float)(i * ST - R);
                const float wx = fmaf(h00, ox, bx);
                const float wy = fmaf(h10, ox, by);
                const float wz = fmaf(h20, ox, bz);
                const float rw = __builtin_amdgcn_rcpf(wz);
                const float u = wx * rw, w = wy * rw;
                // (a wrapped sum lands far outside [0, umax], as any invalid tap)
                const int ix = (int)((unsigned)bu + (unsigned)cvt_flr(u));
                const int iy = (int)((unsigned)bv + (unsigned)cvt_flr(w));
                au[t] = __builtin_amdgcn_fractf(u);
                aw[t] = __builtin_amdgcn_fractf(w);
                // |w_z| guard and 0 <= u < W-1, 0 <= v < H-1 (:289-295); an
                // invalid tap's load goes nowhere and reads zeros (so sval = 0)
                okv[t] = !MASKED || ((!ZCHK || fabsf(wz) >= 1e-8f) & ((unsigned)ix <= umax) &
                                     ((unsigned)iy <= vmax));
                idx[t] = img.index(ix, iy, okv[t]);
                if (!kBurst) {
                    q[t] = img.load(idx[t]);
                    rv[t] = lrow[i * ST];
                }
            }
            if (kBurst) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < C; ++t) q[t] = img.load(idx[t]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < C; ++t) rv[t] = lrow[(t + F < NT ? t + F : t + F - NT) * ST];
            }
#pragma unroll
            for (int t = 0; t < C; ++t) {
                const int ir = i0 + t;
                if (ir >= NT) break;
                const bool ok = okv[t];
                const float sraw = SrcImage<STORE>::lerp(q[t], au[t], aw[t]);
                float r = rv[t];
                float sval;
                if (MASKED) {
                    // an invalid tap read zeros; before the first valid tap s0
                    // stays 0, at it s0 becomes that tap's sample
                    s0 = have ? s0 : sraw;
                    have = have || ok;
                    sval = ok ? sraw - s0 : 0.0f;
                    r = ok ? r : 0.0f;
                    cnt += ok ? 1 : 0;
                } else {
                    if (ir == 0) s0 = jr == 0 ? sraw : s0;
                    sval = sraw - s0;
                }
                if (MASKED) {
                    sr += r;
                    srr = fmaf(r, r, srr);
                }
                ss += sval;
                sss = fmaf(sval, sval, sss);
                srs = fmaf(r, sval, srs);
            }
            // (left to itself the compiler moves a chunk's loads among the last
            // one's samples, until each is waited for by itself)
            if (C < NT) __builtin_amdgcn_sched_barrier(0);
        }
    }
    m.sr = MASKED ? sr : wr.sr;
    m.srr = MASKED ? srr : wr.srr;
    m.ss = ss; m.sss = sss; m.srs = srs;
    m.cnt = MASKED ? cnt : NT * NT;
}

// ---------------------------------------------------------------------------
// Cost of one candidate plane (d, n) at pixel (x, y): patchmatch_mvs.cu:222-343.
// lwin points at the pixel's window top-left tap in the LDS reference tile.
// (rx, ry, rz) is the unnormalised ray K^-1 [x, y, 1] in FP64.
//
// Warp: w(p) = H p with H = A + b g^T, g = K^-T n / (n.P) (the reference's
// q + b * factor, :280-292, in closed form).  The window centre w(x, y) and
// the columns of H are formed in FP64; the taps are w(x, y) + dx h0 + dy h1
// in FP32 with |dx|, |dy| <= 5, so the coordinates are accurate to the FP32
// representation of w even for grazing planes.
// ---------------------------------------------------------------------------
// The candidate's part of the homography: g, and g.p at the window centre.
struct CandPlane {
    double g0, g1, g2, gc;
};

// False where n.P is too small to divide by: the candidate's cost is 2.
__device__ __forceinline__ bool cand_plane(const DevView& v, int x, int y, double rx, double ry,
                                           double rz, float d, float nx, float ny, float nz,
                                           CandPlane& g)
{
    const double dd = d, dnx = nx, dny = ny, dnz = nz;
    const double nP = dd * fma(dnx, rx, fma(dny, ry, dnz * rz));
    if (fabs(nP) < 1e-8) return false;
    const double inv = 1.0 / nP;
    const double* ki = v.kinv_d;
    // g = K^-T n / (n.P): the reference's factor(p) = g.p
    g.g0 = fma(ki[0], dnx, fma(ki[3], dny, ki[6] * dnz)) * inv;
    g.g1 = fma(ki[1], dnx, fma(ki[4], dny, ki[7] * dnz)) * inv;
    g.g2 = fma(ki[2], dnx, fma(ki[5], dny, ki[8] * dnz)) * inv;
    const double X = x, Y = y;
    g.gc = fma(g.g0, X, fma(g.g1, Y, g.g2));   // factor at the window centre
    return true;
}

// Cost 1 - NCC of one candidate plane against source s.
template <int NT, int ST, int STORE, int C, bool BURST = false>
__device__ __forceinline__ float source_cost(const DevView& v, int s,
                                             const float* __restrict__ lwin, int lp,
                                             const WinRef& wr, int x, int y, const CandPlane& g)
{
    constexpr int R = (NT - 1) * ST / 2;
    constexpr int kMinCount = (NT * NT) / 2;
    constexpr bool kLocalCoords = NT * NT <= HP3D_LOCAL_TAPS;
    const double g0 = g.g0, g1 = g.g1, gc = g.gc;
    const double X = x, Y = y;
    const unsigned umax = (unsigned)(v.W - 2), vmax = (unsigned)(v.H - 2);
    constexpr float kShrink = 0.99999904632568359375f;   // 1 - 2^-20
    const float Wq = (float)(v.W - 1) * kShrink, Hq = (float)(v.H - 1) * kShrink;
    const double* A = v.src[s].A;
    const double* b = v.src[s].b;
    // centre of the window and the two tap-step columns of H
    const float cx = (float)fma(b[0], gc, fma(A[0], X, fma(A[1], Y, A[2])));
    const float cy = (float)fma(b[1], gc, fma(A[3], X, fma(A[4], Y, A[5])));
    const float cz = (float)fma(b[2], gc, fma(A[6], X, fma(A[7], Y, A[8])));
    const float h00 = (float)fma(b[0], g0, A[0]), h01 = (float)fma(b[0], g1, A[1]);
    const float h10 = (float)fma(b[1], g0, A[3]), h11 = (float)fma(b[1], g1, A[4]);
    const float h20 = (float)fma(b[2], g0, A[6]), h21 = (float)fma(b[2], g1, A[7]);
    const SrcImage<STORE> img(v, s);

    // Small windows' taps relative to an integer base (bu, bv) near the
    // centre's source position: the base comes out of the centre and the
    // columns in FP64 (u - bu = (w_x - bu w_z) / w_z, still affine in the
    // tap offset over w_z), so the taps' FP32 arithmetic works on u - bu,
    // a few pixels, and rounds to ~ulp(R) instead of ~ulp(u) (1e-5 px at
    // u ~ 100), an error a 3x3 window's NCC amplifies past 1e-4 of cost.
    // A centre that projects beyond 2^22 pixels keeps the base 0.
    float tx = cx, ty = cy, t00 = h00, t01 = h01, t10 = h10, t11 = h11;
    int bu = 0, bv = 0;
    if constexpr (kLocalCoords) {
        const float rc = __builtin_amdgcn_rcpf(cz);
        const float pu = cx * rc, pv = cy * rc;
        bu = fabsf(pu) < 4194304.0f ? (int)rintf(pu) : 0;
        bv = fabsf(pv) < 4194304.0f ? (int)rintf(pv) : 0;
        const double nu = -(double)bu, nv = -(double)bv;
        const double CZ = fma(b[2], gc, fma(A[6], X, fma(A[7], Y, A[8])));
        const double H20 = fma(b[2], g0, A[6]), H21 = fma(b[2], g1, A[7]);
        tx = (float)fma(nu, CZ, fma(b[0], gc, fma(A[0], X, fma(A[1], Y, A[2]))));
        t00 = (float)fma(nu, H20, fma(b[0], g0, A[0]));
        t01 = (float)fma(nu, H21, fma(b[0], g1, A[1]));
        ty = (float)fma(nv, CZ, fma(b[1], gc, fma(A[3], X, fma(A[4], Y, A[5]))));
        t10 = (float)fma(nv, H20, fma(b[1], g0, A[3]));
        t11 = (float)fma(nv, H21, fma(b[1], g1, A[4]));
    }

    // The unmasked tap loop when every lane's window is inside the
    // source image (windows with w_z < 0 throughout take the masked
    // loop, which gives the same result).
    const bool inside = window_inside(cx, cy, cz, h00, h01, h10, h11, h20, h21, (float)R,
                                      Wq, Hq);
    // Where the masked loop has a third form without the per-tap |w_z| test: it
    // gains 2 % with FP16 storage and 1-3 % with FP32 at stride 1 (1280x960, 8
    // sources, 11 x 11 taps: 1.84 -> 1.81 ms a half-pass; 800x600, 5 x 5: 86.8 ->
    // 84.8 us), and loses 2 % with FP32 at stride 2 and 3 % in the 11-tap FP32 cost.
    constexpr bool kZClear = STORE == kStoreF16 || (ST == 1 && (NT <= 7 || C < NT));
    TapSums m;
    // No tap of any lane's window in the image: the cost is that of no sample.
    // (9 % of the wave evaluations of a 4-source 30-degree arc, image-edge
    // bands that the outer sources do not see, otherwise run the masked loop
    // for nothing.)  Not for windows of up to 3 taps a row, whose loop is hardly
    // longer than the test: it took them 10 to 17 registers, with FP16 planes or
    // 2 x 2 taps the fifth wave (two 640x480 views, 2 sources, 8 iterations, 2 x 2
    // FP32: 0.546 ms without, 0.694 with; 3 x 3 FP16 0.666, 0.788).
    if (NT >= kOutsideTaps && !__all(inside)) {
        bool outside = window_outside(cx, cy, cz, h00, h01, h10, h11, h20, h21, (float)R,
                                      (float)v.W, (float)v.H);
        if constexpr (kLocalCoords)
            outside = outside && fabsf((float)bu) <= kOutsideBase && fabsf((float)bv) <= kOutsideBase;
        if (__all(outside)) return 2.0f;
    }
    if (__all(inside)) {
        tap_window<NT, ST, STORE, false, true, C, BURST>(img, lwin, lp, tx, ty, cz, t00, t01, t10,
                                                   t11, h20, h21, umax, vmax, wr, m, bu, bv);
    } else if (kZClear && __all(z_clear(cz, h20, h21, (float)R))) {
        tap_window<NT, ST, STORE, true, false, C, BURST>(img, lwin, lp, tx, ty, cz, t00, t01, t10,
                                                   t11, h20, h21, umax, vmax, wr, m, bu, bv);
    } else {
        tap_window<NT, ST, STORE, true, true, C, BURST>(img, lwin, lp, tx, ty, cz, t00, t01, t10,
                                                  t11, h20, h21, umax, vmax, wr, m, bu, bv);
    }
    const int cnt = m.cnt;
    const float sr = m.sr, ss = m.ss, srr = m.srr, sss = m.sss, srs = m.srs;
    float c = 2.0f;
    if (cnt >= kMinCount) {
        // the products of two floats are exact in FP64, so each difference
        // rounds once with or without the FMA
        const double fc = (double)cnt;
        const double num = fma(fc, (double)srs, -((double)sr * (double)ss));
        const double dr = fma(fc, (double)srr, -((double)sr * (double)sr));
        const double ds = fma(fc, (double)sss, -((double)ss * (double)ss));
        if (!(dr < (double)v.den_eps) && !(ds < (double)v.den_eps)) {
            // dr, ds >= den_eps (~0.065): far from the denormal range,
            // where rsqrtf would first rescale, so the bare v_rsq_f32
            float ncc = (float)num * __builtin_amdgcn_rsqf((float)dr * (float)ds);
            ncc = fmaxf(-1.0f, fminf(1.0f, ncc));
            c = 1.0f - ncc;
        }
    }
    return c;
}

// The ascending list of a candidate's smallest source costs: 3 entries
// suffice when at most 3 are averaged (the reference's top-3), else 8.
struct TopCosts {
    float top[kMaxTopK];
    __device__ __forceinline__ TopCosts()
    {
#pragma unroll
        for (int k = 0; k < kMaxTopK; ++k) top[k] = 2.0f;
    }
    // entry k becomes the median of c and its old neighbours k - 1 and k: c if
    // it falls between them, the lower one if c pushes it up, else unchanged
    __device__ __forceinline__ void insert(float c, bool small_k)
    {
        if (small_k) {
#pragma unroll
            for (int k = 2; k > 0; --k) top[k] = __builtin_amdgcn_fmed3f(c, top[k - 1], top[k]);
        } else {
#pragma unroll
            for (int k = kMaxTopK - 1; k > 0; --k)
                top[k] = __builtin_amdgcn_fmed3f(c, top[k - 1], top[k]);
        }
        top[0] = fminf(c, top[0]);
    }
    // What mean() cannot be below once one more cost (>= 0) is inserted: the same
    // sum, of entries none of which is larger, and rounding keeps that order.
    // Only for means of two or three.
    __device__ __forceinline__ float bound(const DevView& v) const
    {
        const int k = v.top_k < v.S ? v.top_k : v.S;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (i < k - 1) sum += top[i];
        return sum / (float)k;
    }
    __device__ __forceinline__ float mean(const DevView& v) const
    {
        const int k = v.top_k < v.S ? v.top_k : v.S;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kMaxTopK; ++i)
            if (i < k) sum += top[i];
        return sum / (float)k;
    }
};

template <int NT, int ST, int STORE, int C, bool BURST = false>
__device__ __forceinline__ float cand_cost(const DevView& v, const float* __restrict__ lwin,
                                           int lp, const WinRef& wr, int x, int y, double rx,
                                           double ry, double rz, float d, float nx, float ny,
                                           float nz)
{
    CandPlane g;
    if (!cand_plane(v, x, y, rx, ry, rz, d, nx, ny, nz, g)) return 2.0f;
    TopCosts t;
    const bool small_k = v.top_k <= 3;   // wave-uniform
    for (int s = 0; s < v.S; ++s)
        t.insert(source_cost<NT, ST, STORE, C, BURST>(v, s, lwin, lp, wr, x, y, g), small_k);
    return t.mean(v);
}

// ---------------------------------------------------------------------------
// Reference tile staging: rows y0-R .. y0+TY-1+R, columns 2*bx*TX-R ..
// 2*bx*TX+2*TX-1+R, clamped to the image (texture clamp, :807-808).
// ---------------------------------------------------------------------------
template <int R, int STORE, int TX, int TY>
struct TileGeom {
    static constexpr int LW = 2 * TX + 2 * R;   // LDS tile width (pixels)
    static constexpr int LH = TY + 2 * R;       // LDS tile height
    static constexpr int LP = LW + 1;           // LDS row pitch
};

// Tile (bx, by) covers compacted columns bx*TX .. bx*TX+TX-1 (pixel columns
// 2*bx*TX .. 2*bx*TX+2*TX-1) of rows by*TY .. by*TY+TY-1.
template <int R, int STORE, int TX, int TY>
__device__ __forceinline__ void stage_ref_tile(const DevView& v, float* tile, int bx, int by,
                                               int threads = TX * TY)
{
    using G = TileGeom<R, STORE, TX, TY>;
    const int X0 = 2 * bx * TX - R;
    const int Y0 = by * TY - R;
    for (int k = threadIdx.x; k < G::LW * G::LH; k += threads) {
        const int ly = k / G::LW, lx = k - ly * G::LW;
        const int gx = min(max(X0 + lx, 0), v.W - 1);
        const int gy = min(max(Y0 + ly, 0), v.H - 1);
        tile[ly * G::LP + lx] = load_plain<STORE>(v.ref_plain, gy * v.pitch_plain + gx);
    }
    __syncthreads();
}

// Random initial hypothesis of pixel (x, y): init_depth_normal_kernel (:164-216).
__device__ __forceinline__ float4 init_hyp(const DevView& v, int x, int y, uint64_t seed)
{
    uint32_t c0 = (uint32_t)(y * v.W + x), c1 = 0u, c2 = 0u, c3 = kDomainInit;
    philox(c0, c1, c2, c3, (uint32_t)seed, (uint32_t)(seed >> 32));
    const float d = v.dmin + u01(c0) * (v.dmax - v.dmin);
    float rx, ry, rz;
    unit_ray(v.kinv, x, y, rx, ry, rz);
    const float theta = u01(c1) * 6.28318530f;
    const float cos_phi = u01(c2);
    const float sin_phi = sqrtf(1.0f - cos_phi * cos_phi);
    float nx = sin_phi * (float)cos((double)theta);
    float ny = sin_phi * (float)sin((double)theta);
    float nz = cos_phi;
    if (nx * rx + ny * ry + nz * rz > 0.0f) { nx = -nx; ny = -ny; nz = -nz; }
    const float nlen = sqrtf(nx * nx + ny * ny + nz * nz);
    if (nlen > 1e-12f) { nx = nx / nlen; ny = ny / nlen; nz = nz / nlen; }
    return make_float4(d, nx, ny, nz);
}

// Cost of the current hypothesis of the colour-`parity` pixel of lane (tx, ty)
// in tile (bx, by); returns false if the lane has no pixel.
template <int NT, int ST, int STORE, int TX, int TY, int C = kCostChunk<NT>, bool COH = false>
__device__ __forceinline__ bool cost_pixel(const DevView& v, const float* tile, int bx, int by,
                                           int tx, int ty, int parity)
{
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    const int i = bx * TX + tx;
    const int y = by * TY + ty;
    const int x = 2 * i + ((y + parity) & 1);
    if (y >= v.H || x >= v.W) return false;
    const float* lwin = tile + ty * G::LP + (x - 2 * bx * TX);
    double rx, ry, rz;
    ray_fp64(v.kinv_d, x, y, rx, ry, rz);
    const int p = y * v.Wc + i;
    const float4 h = StateIO<COH>::ld4(v.hyp[parity], p);
    const WinRef wr = window_ref_sums<NT, ST>(lwin, G::LP);
    StateIO<COH>::st1(v.cost[parity], p,
                      cand_cost<NT, ST, STORE, C>(v, lwin, G::LP, wr, x, y, rx, ry, rz, h.x, h.y,
                                                  h.z, h.w));
    return true;
}

// Orders a wave's accesses to LDS that no other wave touches: the hardware
// keeps their order, the fence keeps the compiler's.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// LDS scratch of a workgroup of T threads in a pass: the list of the neighbour
// candidates that must be evaluated (owner thread | candidate << 10, at most 4
// per thread), their hypotheses (by candidate, then owner: each is loaded
// once, by its owner, and read from here by the lane that evaluates it and by
// the owner when it accepts it), their costs by list position, the owners'
// reference sums, and the counts that place entries in the list.
template <int T> struct PassXchg {
    static_assert(T % 64 == 0 && T <= 1024, "whole waves, 10 bits of owner thread");
    unsigned short item[4 * T];
    float4 hyp[4 * T];
    float cost[4 * T];
    WinRef wref[T];
    int hist[T];        // 64 depth buckets per wave
    int wsum[T / 64];   // entries per wave
    int rsum[2][T / 64];   // refinement candidates per wave that need their last source
};

// Where halfpass_pixel pools the refinement candidates' last source (at its
// loop): a bound needs a mean over two or three of at least two sources, and from
// the seventh iteration on the candidates lie so near the current hypothesis that
// few are rejected before it (640x480, 4 sources, 6 x 6 taps, the first step's
// candidates: 59, 74, 67 and 41 % in the first, second, fourth and sixth
// iteration, 12 % in the eighth).
__host__ __device__ __forceinline__ bool pool_refinement(int S, int top_k, int iteration)
{
    return S >= 2 && top_k >= 2 && top_k <= 3 && iteration < 6;
}

// Depth buckets of a wave's counting sort: inverse depth (disparity) over the
// view's range.
struct DepthBuckets {
    float ilo, iscale;
    __device__ __forceinline__ DepthBuckets(float dmin, float dmax)
        : ilo(1.0f / dmax), iscale(64.0f / (1.0f / dmin - ilo)) {}
    __device__ __forceinline__ int of(float d) const
    {
        const int b = (int)((1.0f / d - ilo) * iscale);
        return b < 0 ? 0 : (b > 63 ? 63 : b);
    }
};

// Counts to places: on return hist[b] is the sum of the wave's counts below b.
__device__ __forceinline__ void scan_buckets(int* hist, int lane)
{
    wave_lds_order();
    const int cnt = hist[lane];
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
    }
    wave_lds_order();
    hist[lane] = incl - cnt;
    wave_lds_order();
}

// Cost of the current hypotheses of colour `parity` at this workgroup's
// pixels (compute_ncc_cost_kernel, patchmatch_mvs.cu:349-513), evaluated in
// inverse-depth order within each wave: the hypotheses are random, so each
// lane's windows would gather from an unrelated part of every source; a
// counting sort of the wave's hypotheses by inverse depth (disparity) hands
// lane k the k-th, so a wave's gathers fall in a narrower band of each
// source.  (Sorted over the whole workgroup the bands are narrower still, but
// a wave's pixels spread over the tile: 0.149 -> 0.155 ms a colour at
// 1600x1200.)  Any lane can evaluate any pixel's candidate (the whole window
// tile is in LDS) and a cost is a pure function of the pixel and the
// hypothesis, so the result is the same as one lane per pixel.
template <int NT, int ST, int STORE, int TX, int TY, bool COH = false>
__device__ __forceinline__ void cost_tile_sorted(const DevView& v, const float* tile, int bx,
                                                 int by, int tx, int ty, int parity,
                                                 PassXchg<TX * TY>& xc)
{
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    using IO = StateIO<COH>;
    const int t = threadIdx.x, lane = t & 63, wave0 = t & ~63;
    const int i = bx * TX + tx, y = by * TY + ty;
    const int x = 2 * i + ((y + parity) & 1);
    const bool active = y < v.H && x < v.W;
    float4 h = make_float4(0.f, 0.f, 0.f, 0.f);
    if (active) h = IO::ld4(v.hyp[parity], y * v.Wc + i);
    int* hist = xc.hist + wave0;
    hist[lane] = 0;
    wave_lds_order();
    int bk = 0, rk = 0;
    if (active) {
        bk = DepthBuckets(v.dmin, v.dmax).of(h.x);
        rk = atomicAdd(&hist[bk], 1);
    }
    scan_buckets(hist, lane);
    if (active) {
        const int slot = wave0 + hist[bk] + rk;
        xc.item[slot] = (unsigned short)t;
        xc.hyp[slot] = h;
    }
    const int total = __popcll(__ballot(active));
    wave_lds_order();
    if (lane < total) {
        const int t_o = xc.item[t];
        const float4 hh = xc.hyp[t];
        const int tx_o = t_o % TX, ty_o = t_o / TX;
        const int i_o = bx * TX + tx_o, y_o = by * TY + ty_o;
        const int x_o = 2 * i_o + ((y_o + parity) & 1);
        const float* lwin = tile + ty_o * G::LP + (x_o - 2 * bx * TX);
        const WinRef wr = window_ref_sums<NT, ST>(lwin, G::LP);
        double rx, ry, rz;
        ray_fp64(v.kinv_d, x_o, y_o, rx, ry, rz);
        IO::st1(v.cost[parity], y_o * v.Wc + i_o,
                cand_cost<NT, ST, STORE, kCostChunk<NT>, (NT >= 11 && STORE == kStoreF32)>(
                    v, lwin, G::LP, wr, x_o, y_o, rx, ry, rz, hh.x, hh.y, hh.z, hh.w));
    }
}

// A refinement candidate: the current hypothesis moved by the draw's four
// words within the given ranges, its normal normalised and camera-facing
// (propagate_and_refine_kernel, :610-640).
__device__ __forceinline__ float4 refine_cand(const float4& best, const uint4& w,
                                              float depth_range, float normal_range, float dmin,
                                              float dmax, float ux, float uy, float uz)
{
    const float rand_d = u01(w.x) * 2.0f - 1.0f;
    float cd = best.x + rand_d * depth_range;
    cd = fmaxf(dmin, fminf(dmax, cd));
    float cnx = best.y + (u01(w.y) * 2.0f - 1.0f) * normal_range;
    float cny = best.z + (u01(w.z) * 2.0f - 1.0f) * normal_range;
    float cnz = best.w + (u01(w.w) * 2.0f - 1.0f) * normal_range;
    const float nlen = sqrtf(cnx * cnx + cny * cny + cnz * cnz);
    if (nlen > 1e-12f) { cnx = cnx / nlen; cny = cny / nlen; cnz = cnz / nlen; }
    if (cnx * ux + cny * uy + cnz * uz > 0.0f) { cnx = -cnx; cny = -cny; cnz = -cnz; }
    return make_float4(cd, cnx, cny, cnz);
}

// One pixel of a red (parity 0) or black (parity 1) half-pass:
// propagate_and_refine_kernel (:519-655).  Candidates L, R, U, D from the
// other colour plane, then two random refinements with ranges
// (dmax-dmin)/2 * 0.6^iter and 0.6^iter, halved per step.  Strict '<'
// acceptance throughout.
//
// A neighbour candidate that is bit-identical to the pixel's own hypothesis,
// or to an earlier valid candidate, cannot be accepted: its cost is the same
// deterministic function of (pixel, hypothesis), and bc is already at most
// that cost.  Once propagation has spread planes, 40-60 % of the neighbour
// candidates are such repeats, but rarely all 64 lanes of a wave at once.  So
// the workgroup lists the candidates its lanes still need (also leaving out
// neighbours unchanged since this pixel's previous pass, see below), any
// lane evaluates any
// pixel's candidate (all windows of the workgroup are in LDS), and each
// owner then applies the costs in L, R, U, D order.  The result is the one
// the plain per-lane loop gives, with fewer evaluation rounds.
// Every thread of the workgroup must call this (it synchronises the group),
// with the same pool (see pool_refinement).
template <int NT, int ST, int STORE, int TX, int TY, bool COH = false>
__device__ __forceinline__ void halfpass_pixel(const DevView& v, const float* tile, int bx, int by,
                                               int tx, int ty, int iteration, int parity,
                                               uint64_t pass_seed, PassXchg<TX * TY>& xc,
                                               bool pool = false)
{
    constexpr int R = (NT - 1) * ST / 2, T = TX * TY;
    using G = TileGeom<R, STORE, TX, TY>;
    using IO = StateIO<COH>;
    const int t = threadIdx.x, lane = t & 63, wave0 = t & ~63;
    const int i = bx * TX + tx;
    const int y = by * TY + ty;
    const int o = (y + parity) & 1;
    const int x = 2 * i + o;
    const bool active = y < v.H && x < v.W;
    const float* lwin = tile + ty * G::LP + (x - 2 * bx * TX);
    const float dmin = v.dmin, dmax = v.dmax;
    const int Wc = v.Wc;
    float4* own = v.hyp[parity];
    const float4* oth = v.hyp[parity ^ 1];
    const int p = y * Wc + i;
    // neighbour positions in the other plane: L = i+o-1, R = i+o (row y),
    // U, D = i (rows y-1, y+1)
    auto nb = [&](int k, int pp, int oo) {
        return k == 0 ? pp + oo - 1 : k == 1 ? pp + oo : k == 2 ? pp - Wc : pp + Wc;
    };
    auto same = [](const float4& a, const float4& b) {
        return __float_as_uint(a.x) == __float_as_uint(b.x) &&
               __float_as_uint(a.y) == __float_as_uint(b.y) &&
               __float_as_uint(a.z) == __float_as_uint(b.z) &&
               __float_as_uint(a.w) == __float_as_uint(b.w);
    };

    float4 best = make_float4(0.f, 0.f, 0.f, 0.f);
    float bc = 2.0f;
    bool changed = false;
    unsigned need = 0;   // bit k: neighbour k has to be evaluated
    float hd[4] = {0.f, 0.f, 0.f, 0.f};   // the candidates' depths
    if (active) {
        best = IO::ld4(own, p);
        bc = IO::ld1(v.cost[parity], p);
        // From the second iteration of a solve on, this pixel evaluated its
        // neighbours' hypotheses one iteration ago; a neighbour that did not
        // change since (its flag from the other colour's last half-pass)
        // still holds that hypothesis, whose cost was then >= bc, and bc has
        // only decreased: it cannot be accepted now.
        const bool seen = iteration > v.first_iteration;
        const unsigned char* chg_oth = v.chg[parity ^ 1];
        float4 h[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool has = k == 0 ? x >= 1 : k == 1 ? x + 1 < v.W : k == 2 ? y >= 1 : y + 1 < v.H;
            ok[k] = false;
            h[k] = best;
            bool stale = false;
            if (has) {
                const int q = nb(k, p, o);
                h[k] = IO::ld4(oth, q);
                ok[k] = !(h[k].x < dmin || h[k].x > dmax);
                stale = seen && IO::ldb(chg_oth, q) == 0;
            }
            bool n = ok[k] && !stale && !same(h[k], best);
#pragma unroll
            for (int j = 0; j < k; ++j) n = n && !(ok[j] && same(h[j], h[k]));
            need |= (unsigned)n << k;
            hd[k] = h[k].x;
            if (n) xc.hyp[t + k * T] = h[k];
        }
    }
    const WinRef wr = window_ref_sums<NT, ST>(lwin, G::LP);
    xc.wref[t] = wr;

    // The workgroup's list, ordered by owner thread, then candidate: a round of
    // 64 items then covers neighbouring pixels whose candidates project to
    // nearly the same source rows and columns, so its gathers touch far
    // fewer 64-B segments than 64 pixels' worth would.  The waves take its
    // rounds in turn: per wave, the last round would on average be half empty,
    // half of the 3 to 4 rounds a converged pass has (1600x1200, 4 sources,
    // stride 2: 0.446 -> 0.427 ms a half-pass; 1280x960, 8 sources, stride 1:
    // 1.77 -> 1.68 ms; with 512 threads 3 % slower again).
    const unsigned long long below = (1ull << lane) - 1ull;
    int slot[4];
    int base = 0, count = 0;   // entries of the lanes below this one, of the wave
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned long long m = __ballot((need >> k) & 1u);
        base += __popcll(m & below);
        count += __popcll(m);
    }
    if (lane == 0) xc.wsum[t >> 6] = count;
    bool sorted = false;
#if HP3D_BUCKET
    if (NT < 9 && iteration < v.first_iteration + HP3D_BUCKET) {
        // First iteration: the neighbours hold random, unrelated depths, so
        // owner order does not cluster the gathers.  Order each wave's entries
        // by inverse depth (disparity) instead (the order within a bucket does
        // not matter), so a round's windows lie in a narrower band of every
        // source.  (+1.4 % on 6x6-tap windows; with 11x11 windows it measured
        // slower, and so did sorting over the workgroup: 0.744 -> 0.818 ms.)
        int* hist = xc.hist + wave0;
        const DepthBuckets db(dmin, dmax);
        hist[lane] = 0;
        wave_lds_order();
        int bk[4], rk[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            bk[k] = 0;
            rk[k] = 0;
            if ((need >> k) & 1u) {
                bk[k] = db.of(hd[k]);
                rk[k] = atomicAdd(&hist[bk[k]], 1);
            }
        }
        scan_buckets(hist, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) slot[k] = hist[bk[k]] + rk[k];
        sorted = true;
    }
#endif
    if (!sorted) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            slot[k] = base;
            base += (need >> k) & 1u;
        }
    }
    __syncthreads();
    int first = 0, total = 0;   // this wave's first entry, the workgroup's entries
#pragma unroll
    for (int w = 0; w < T / 64; ++w) {
        const int c = xc.wsum[w];
        if (w < (t >> 6)) first += c;
        total += c;
    }
    total = __builtin_amdgcn_readfirstlane(total);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        slot[k] += first;
        if ((need >> k) & 1u) xc.item[slot[k]] = (unsigned short)(t | (k << 10));
    }
    __syncthreads();
    for (int g0 = __builtin_amdgcn_readfirstlane(wave0); g0 < total; g0 += T) {
        const int g = g0 + lane;
        if (g < total) {
            const unsigned it = xc.item[g];
            const int t_o = it & 1023;
            const int tx_o = t_o % TX, ty_o = t_o / TX;
            const int i_o = bx * TX + tx_o, y_o = by * TY + ty_o;
            const int o_o = (y_o + parity) & 1, x_o = 2 * i_o + o_o;
            const float4 h = xc.hyp[t_o + (int)(it >> 10) * T];
            double rx, ry, rz;
            ray_fp64(v.kinv_d, x_o, y_o, rx, ry, rz);
            xc.cost[g] = cand_cost<NT, ST, STORE, kPassChunk<NT>>(
                v, tile + ty_o * G::LP + (x_o - 2 * bx * TX), G::LP, xc.wref[t_o], x_o, y_o, rx,
                ry, rz, h.x, h.y, h.z, h.w);
        }
    }
    __syncthreads();
    if (!pool && !active) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!((need >> k) & 1u)) continue;
        const float c = xc.cost[slot[k]];
        if (c < bc) { bc = c; best = xc.hyp[t + k * T]; changed = true; }
    }

    float depth_range = (dmax - dmin) * 0.5f;
    float normal_range = 1.0f;
    for (int it = 0; it < iteration; ++it) { depth_range *= 0.6f; normal_range *= 0.6f; }
    const uint32_t idx = (uint32_t)(y * v.W + x);
    if (pool) {
        // A candidate whose mean without its last source cannot be below the
        // current cost is not accepted whatever that source says.  After the
        // other sources the workgroup lists the lanes that still need it, and
        // where they fit into fewer rounds than it has waves, wave w evaluates the
        // last source of entries 64 w .. 64 w + 63.  Rejected or not, the costs
        // that are compared are those of the plain loop below.  (Half-passes of
        // 8-iteration solves: 2400x1800, 4 sources, 6 x 6 taps, FP16 879 -> 838 us;
        // 1280x960, 8 sources, 11 x 11, FP32 1610 -> 1567; 3 sources, 7 x 7 286 ->
        // 276.  The neighbours' list the same way gained nothing: fewer of them are
        // rejected, and every group of T entries waits for its slowest wave.)
#pragma unroll 1
        for (int step = 0; step < 2; ++step) {
            // (what can be read from LDS or formed again is: held in registers
            // through the sources, the candidate, its pixel and its window sums took
            // the 6-tap and 7-tap FP32 kernels past 128, with two spilled to scratch)
            int te = t;   // the owner of the candidate that this lane evaluates
            CandPlane g;
            bool live = active;
            if (active) {
                uint32_t c0 = idx, c1 = (uint32_t)iteration, c2 = (uint32_t)step, c3 = kDomainRefine;
                philox(c0, c1, c2, c3, (uint32_t)pass_seed, (uint32_t)(pass_seed >> 32));
                float ux, uy, uz;
                unit_ray(v.kinv, x, y, ux, uy, uz);
                const float4 cand = refine_cand(best, make_uint4(c0, c1, c2, c3), depth_range,
                                                normal_range, dmin, dmax, ux, uy, uz);
                xc.hyp[t] = cand;
                double rx, ry, rz;
                ray_fp64(v.kinv_d, x, y, rx, ry, rz);
                live = cand_plane(v, x, y, rx, ry, rz, cand.x, cand.y, cand.z, cand.w, g);
            }
            bool run = live, pooled = false;
            int place = 0;
            TopCosts top;
            for (int s = 0; s < v.S; ++s) {
                if (s == v.S - 1) {
                    live = live && top.bound(v) < bc;
                    const unsigned long long m = __ballot(live);
                    if (lane == 0) xc.rsum[step][t >> 6] = __popcll(m);
                    __syncthreads();
                    int all = 0;
                    place = __popcll(m & below);
#pragma unroll
                    for (int w = 0; w < T / 64; ++w) {
                        const int c = xc.rsum[step][w];
                        if (w < (t >> 6)) place += c;
                        all += c;
                    }
                    all = __builtin_amdgcn_readfirstlane(all);
                    pooled = all <= T - 64;
                    run = live;
                    if (pooled) {
                        if (live) xc.item[place] = (unsigned short)t;
                        __syncthreads();
                        run = t < all;
                        if (run) {
                            te = xc.item[t];
                            const int ye = by * TY + te / TX;
                            const int xe = 2 * (bx * TX + te % TX) + ((ye + parity) & 1);
                            const float4 h = xc.hyp[te];
                            double qx, qy, qz;
                            ray_fp64(v.kinv_d, xe, ye, qx, qy, qz);
                            cand_plane(v, xe, ye, qx, qy, qz, h.x, h.y, h.z, h.w, g);
                        }
                    }
                }
                if (run) {
                    const int ye = by * TY + te / TX;
                    const int xe = 2 * (bx * TX + te % TX) + ((ye + parity) & 1);
                    const float c = source_cost<NT, ST, STORE, kPassChunk<NT>>(
                        v, s, tile + te / TX * G::LP + (xe - 2 * bx * TX), G::LP, xc.wref[te], xe,
                        ye, g);
                    if (pooled) xc.cost[t] = c;
                    else top.insert(c, true);
                }
            }
            if (pooled) {
                __syncthreads();
                if (live) top.insert(xc.cost[place], true);
            }
            const float c = top.mean(v);
            if (live && c < bc) { bc = c; best = xc.hyp[t]; changed = true; }
            depth_range *= 0.5f;
            normal_range *= 0.5f;
        }
        if (!active) return;
    } else {
        double rx, ry, rz;
        ray_fp64(v.kinv_d, x, y, rx, ry, rz);
        float ux, uy, uz;
        unit_ray(v.kinv, x, y, ux, uy, uz);
#pragma unroll 1
        for (int step = 0; step < 2; ++step) {
            uint32_t c0 = idx, c1 = (uint32_t)iteration, c2 = (uint32_t)step, c3 = kDomainRefine;
            philox(c0, c1, c2, c3, (uint32_t)pass_seed, (uint32_t)(pass_seed >> 32));
            const float4 cand = refine_cand(best, make_uint4(c0, c1, c2, c3), depth_range,
                                            normal_range, dmin, dmax, ux, uy, uz);
            const float c = cand_cost<NT, ST, STORE, kPassChunk<NT>>(v, lwin, G::LP, wr, x, y, rx, ry, rz, cand.x,
                                                     cand.y, cand.z, cand.w);
            if (c < bc) { bc = c; best = cand; changed = true; }
            depth_range *= 0.5f;
            normal_range *= 0.5f;
        }
    }
    IO::st4(own, p, best);
    IO::st1(v.cost[parity], p, bc);
    IO::stb(v.chg[parity], p, changed ? 1u : 0u);
}

// ---------------------------------------------------------------------------
// The same passes for views of few pixels: a workgroup of up to kMaxSplitWaves
// waves takes the 64 pixels of one colour in a tile (TX * TY = 64), and its
// waves share the evaluations, one (64 candidates, source) at a time.  A
// source's cost is a pure function of (pixel, hypothesis, source) and goes to
// its place in LDS, so the costs, and the means over the smallest of them, are
// the bits one lane per pixel gives.
//
// What bounds such a view is the chain of evaluations that one wave of
// halfpass_pixel does one after another, up to 6 candidates x S sources, while
// most of the 1024 SIMDs have no wave (a 96x72 view has 54).  With a wave per
// source the chain is 4 + 1 + 1 evaluations; with 4 S waves the rounds of
// neighbours run side by side too, and with 3 S the two refinement steps: the
// second is evaluated for both outcomes of the first.
// ---------------------------------------------------------------------------
constexpr int kMaxSplitWaves = 16;

struct SplitXchg {
    unsigned char item[256];               // listed neighbours: owner lane | candidate << 6
    float4 hyp[256];                       // their hypotheses, by the same index
    float cost[kMaxSrc][256];              // source costs by list position
    float cost_r[3][kMaxSrc][64];          // source costs of the refinement candidates
    uint4 rnd[2][64];                      // the refinement steps' Philox words
};

// Mean of the smallest source costs at position g.
template <int N>
__device__ __forceinline__ float split_mean(const DevView& v, const float (*cost)[N], int g)
{
    TopCosts t;
    const bool small_k = v.top_k <= 3;
    for (int s = 0; s < v.S; ++s) t.insert(cost[s][g], small_k);
    return t.mean(v);
}

template <int NT, int ST, int STORE, int TX, int TY>
__device__ __forceinline__ void halfpass_split(const DevView& v, float* tile, int bx, int by,
                                               int iteration, int parity, uint64_t pass_seed,
                                               SplitXchg& xs)
{
    static_assert(TX * TY == 64, "one wave of pixels per tile");
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int waves = (int)blockDim.x >> 6;
    const int tx = lane % TX, ty = lane / TX;
    const int i = bx * TX + tx, y = by * TY + ty;
    const int o = (y + parity) & 1, x = 2 * i + o;
    const bool active = y < v.H && x < v.W;
    const float dmin = v.dmin, dmax = v.dmax;
    const int Wc = v.Wc, p = y * Wc + i;
    auto same = [](const float4& a, const float4& b) {
        return __float_as_uint(a.x) == __float_as_uint(b.x) &&
               __float_as_uint(a.y) == __float_as_uint(b.y) &&
               __float_as_uint(a.z) == __float_as_uint(b.z) &&
               __float_as_uint(a.w) == __float_as_uint(b.w);
    };
    stage_ref_tile<R, STORE, TX, TY>(v, tile, bx, by, (int)blockDim.x);
    if (wave == waves - 1) {
        // the refinement draws depend on no hypothesis
#pragma unroll 1
        for (int step = 0; step < 2; ++step) {
            uint32_t c0 = (uint32_t)(y * v.W + x), c1 = (uint32_t)iteration, c2 = (uint32_t)step;
            uint32_t c3 = kDomainRefine;
            philox(c0, c1, c2, c3, (uint32_t)pass_seed, (uint32_t)(pass_seed >> 32));
            xs.rnd[step][lane] = make_uint4(c0, c1, c2, c3);
        }
    }
    // every wave holds its lane's pixel: which neighbours have to be evaluated
    // (the conditions of halfpass_pixel) and where they are listed
    float4 best = make_float4(0.f, 0.f, 0.f, 0.f);
    float bc = 2.0f;
    unsigned need = 0;
    if (active) {
        const float4* oth = v.hyp[parity ^ 1];
        const unsigned char* chg_oth = v.chg[parity ^ 1];
        best = v.hyp[parity][p];
        bc = v.cost[parity][p];
        const bool seen = iteration > v.first_iteration;
        float4 h[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool has = k == 0 ? x >= 1 : k == 1 ? x + 1 < v.W : k == 2 ? y >= 1 : y + 1 < v.H;
            const int q = k == 0 ? p + o - 1 : k == 1 ? p + o : k == 2 ? p - Wc : p + Wc;
            ok[k] = false;
            h[k] = best;
            bool stale = false;
            if (has) {
                h[k] = oth[q];
                ok[k] = !(h[k].x < dmin || h[k].x > dmax);
                stale = seen && chg_oth[q] == 0;
            }
            bool n = ok[k] && !stale && !same(h[k], best);
#pragma unroll
            for (int j = 0; j < k; ++j) n = n && !(ok[j] && same(h[j], h[k]));
            need |= (unsigned)n << k;
            if (n && wave == 0) xs.hyp[lane | (k << 6)] = h[k];
        }
    }
    const unsigned long long below = (1ull << lane) - 1ull;
    int base = 0, total = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned long long m = __ballot((need >> k) & 1u);
        base += __popcll(m & below);
        total += __popcll(m);
    }
    if (wave == 0) {
        int off = base;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if ((need >> k) & 1u) xs.item[off++] = (unsigned char)(lane | (k << 6));
    }
    __syncthreads();
    const float* lwin = tile + ty * G::LP + (x - 2 * bx * TX);
    const WinRef wr = window_ref_sums<NT, ST>(lwin, G::LP);
    float ux, uy, uz;
    unit_ray(v.kinv, x, y, ux, uy, uz);
    float depth_range = (dmax - dmin) * 0.5f, normal_range = 1.0f;
    for (int it = 0; it < iteration; ++it) { depth_range *= 0.6f; normal_range *= 0.6f; }
    // the refinement candidate of a step from hypothesis h
    auto draw = [&](int step, const float4& h) {
        const float f = step ? 0.5f : 1.0f;
        return refine_cand(h, xs.rnd[step][lane], depth_range * f, normal_range * f, dmin, dmax,
                           ux, uy, uz);
    };
    // phase 0: the listed neighbours, 64 a round; phase 1: the first refinement
    // step and, with the waves for it, the second step from either outcome;
    // phase 2: else the second step
    const bool both = waves >= 3 * v.S;
    bool changed = false;
#pragma unroll 1
    for (int phase = 0; phase < 3; ++phase) {
        const int groups = phase == 0 ? (total + 63) >> 6 : phase == 1 && both ? 3 : 1;
#pragma unroll 1
        for (int u = wave; u < groups * v.S; u += waves) {
            const int r = u / v.S, s = u - r * v.S;
            int ol = lane;
            bool on = active;
            float4 h;
            if (phase == 0) {
                on = r * 64 + lane < total;
                const unsigned it = xs.item[on ? r * 64 + lane : total - 1];
                ol = it & 63;
                h = xs.hyp[it];
            } else {
                h = draw(phase == 2 || r == 1 ? 1 : 0, best);
                if (r == 2) h = draw(1, h);
            }
            const WinRef wro{__shfl(wr.sr, ol, 64), __shfl(wr.srr, ol, 64)};
            if (on) {
                const int tx_o = ol % TX, ty_o = ol / TX;
                const int i_o = bx * TX + tx_o, y_o = by * TY + ty_o;
                const int x_o = 2 * i_o + ((y_o + parity) & 1);
                double rx, ry, rz;
                ray_fp64(v.kinv_d, x_o, y_o, rx, ry, rz);
                CandPlane cp;
                float c = 2.0f;
                if (cand_plane(v, x_o, y_o, rx, ry, rz, h.x, h.y, h.z, h.w, cp))
                    c = source_cost<NT, ST, STORE, kPassChunk<NT>>(
                        v, s, tile + ty_o * G::LP + (x_o - 2 * bx * TX), G::LP, wro, x_o, y_o, cp);
                if (phase == 0) xs.cost[s][r * 64 + lane] = c;
                else xs.cost_r[phase == 2 ? 1 : r][s][lane] = c;
            }
        }
        __syncthreads();
        // the end is one wave's; before it every wave goes on for itself (each
        // needs the hypothesis that the next draw starts from)
        const bool last = phase == 2 || (phase == 1 && both);
        if (last && wave != 0) return;
        if (active) {
            if (phase == 0) {
#pragma unroll 1
                for (int k = 0; k < 4; ++k) {
                    if (!((need >> k) & 1u)) continue;
                    const float c = split_mean(v, xs.cost, base++);
                    if (c < bc) { bc = c; best = xs.hyp[lane | (k << 6)]; changed = true; }
                }
            } else {
                int second = 1;   // where the second step's costs are
                if (phase == 1) {
                    const float c = split_mean(v, xs.cost_r[0], lane);
                    if (c < bc) { bc = c; best = draw(0, best); changed = true; second = 2; }
                }
                if (last) {
                    const float c = split_mean(v, xs.cost_r[phase == 2 ? 1 : second], lane);
                    if (c < bc) { bc = c; best = draw(1, best); changed = true; }
                }
            }
        }
        if (last) break;
    }
    if (!active) return;
    v.hyp[parity][p] = best;
    v.cost[parity][p] = bc;
    v.chg[parity][p] = changed ? 1 : 0;
}

// The initial cost likewise: a wave per source.
template <int NT, int ST, int STORE, int TX, int TY>
__device__ __forceinline__ void cost_split(const DevView& v, float* tile, int bx, int by,
                                           int parity, SplitXchg& xs)
{
    static_assert(TX * TY == 64, "one wave of pixels per tile");
    constexpr int R = (NT - 1) * ST / 2;
    using G = TileGeom<R, STORE, TX, TY>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int waves = (int)blockDim.x >> 6;
    const int tx = lane % TX, ty = lane / TX;
    const int i = bx * TX + tx, y = by * TY + ty;
    const int x = 2 * i + ((y + parity) & 1);
    const bool active = y < v.H && x < v.W;
    stage_ref_tile<R, STORE, TX, TY>(v, tile, bx, by, (int)blockDim.x);
    if (active) {
        const float4 h = v.hyp[parity][y * v.Wc + i];
        const float* lwin = tile + ty * G::LP + (x - 2 * bx * TX);
        const WinRef wr = window_ref_sums<NT, ST>(lwin, G::LP);
        double rx, ry, rz;
        ray_fp64(v.kinv_d, x, y, rx, ry, rz);
        CandPlane cp;
        const bool ok = cand_plane(v, x, y, rx, ry, rz, h.x, h.y, h.z, h.w, cp);
#pragma unroll 1
        for (int s = wave; s < v.S; s += waves) {
            float c = 2.0f;
            if (ok) c = source_cost<NT, ST, STORE, kCostChunk<NT>>(v, s, lwin, G::LP, wr, x, y, cp);
            xs.cost[s][lane] = c;
        }
    }
    __syncthreads();
    if (wave == 0 && active) v.cost[parity][y * v.Wc + i] = split_mean(v, xs.cost, lane);
}

// Row-major outputs of pixel (x, y) from the colour planes.
template <bool COH = false>
__device__ __forceinline__ void emit_pixel(const DevView& v, int x, int y, float* depth,
                                           float* normal, float* cost, float* conf)
{
    const int c = (x + y) & 1, p = y * v.Wc + (x >> 1);
    const size_t q = (size_t)y * v.W + x;
    const float4 h = StateIO<COH>::ld4(v.hyp[c], p);
    if (depth) depth[q] = h.x;
    if (normal) { normal[3 * q] = h.y; normal[3 * q + 1] = h.z; normal[3 * q + 2] = h.w; }
    if (cost || conf) {
        const float k = StateIO<COH>::ld1(v.cost[c], p);
        if (cost) cost[q] = k;
        if (conf) conf[q] = 1.0f - k * 0.5f;   // patchmatch_mvs.cu:1249-1252
    }
}

}  // namespace hp3d
