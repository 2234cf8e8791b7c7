// pm_window.h -- closed-form tests of a whole window: every tap inside the image,
// every tap outside, every |w_z| clear of the guard.  Plain FP32 arithmetic with no
// contraction, so that a host compiler can check the same functions.
#pragma once

namespace hp3d {

// ---------------------------------------------------------------------------
// True if the tap loop, with its FP32 arithmetic, will find every tap of the
// window valid (|w_z| >= 1e-8, 0 <= u < W-1, 0 <= v < H-1), so the unmasked
// loop gives the masked loop's result.  A tap's w = c + ox h_0 + oy h_1 is
// affine in the offset, so over the square |ox|, |oy| <= R its extremes are
// c -/+ R (|a| + |b|): no corners to enumerate.  The conditions used are
//   min w_x > 0, min w_y > 0, min w_z > 1e-8      (then u, v >= 0), and
//   max (w_x - Wq w_z) < 0, max (w_y - Hq w_z) < 0,
// with Wq = (W-1)(1 - 2^-20), so that u = w_x * rcp(w_z) < W-1 even with
// v_rcp_f32's 1-ulp error and the rounding of the product.  Each bound is
// tightened by 2^-21 (8 FP32 rounding units) times the magnitude of the terms
// it is built from (T = |c| + R (|a| + |b|)): a tap's coordinate carries at
// most 2 units of that (two FMAs), the bound's own evaluation at most 4.  So
// the test is exact in what it promises, also for grazing windows where the
// terms nearly cancel.  NaN or infinite inputs fail every comparison.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool window_inside(float cx, float cy, float cz, float h00, float h01,
                                              float h10, float h11, float h20, float h21, float R,
                                              float Wq, float Hq)
{
    constexpr float kE = 4.76837158203125e-07f;   // 2^-21
    const float ax = fabsf(h00) + fabsf(h01), ay = fabsf(h10) + fabsf(h11);
    const float az = fabsf(h20) + fabsf(h21);
    const float Tx = fmaf(R, ax, fabsf(cx)), Ty = fmaf(R, ay, fabsf(cy));
    const float Tz = fmaf(R, az, fabsf(cz));
    const float lox = fmaf(-R, ax, cx), loy = fmaf(-R, ay, cy), loz = fmaf(-R, az, cz);
    const float gx = fmaf(R, fabsf(fmaf(-Wq, h20, h00)) + fabsf(fmaf(-Wq, h21, h01)),
                          fmaf(-Wq, cz, cx));
    const float gy = fmaf(R, fabsf(fmaf(-Hq, h20, h10)) + fabsf(fmaf(-Hq, h21, h11)),
                          fmaf(-Hq, cz, cy));
    return (fmaf(-kE, Tx, lox) >= 0.0f) && (fmaf(-kE, Ty, loy) >= 0.0f) &&
           (fmaf(-kE, Tz, loz) >= 1e-8f) && (fmaf(kE, fmaf(Wq, Tz, Tx), gx) < 0.0f) &&
           (fmaf(kE, fmaf(Hq, Tz, Ty), gy) < 0.0f);
}

// True if every tap of the window provably misses the image, in front of the
// camera and more than a pixel to one side: all u < -1, or all u > W, or the
// same for v and H.  The extremes over the window are affine, as in
// window_inside.  Besides the pixel, each bound is tightened by 2^-21 of
// T_x + (W + 2^17) T_z, which covers the rounding of a tap's coordinate also
// relative to an integer base of up to 2^17 (small windows), and u is compared
// at W (1 + 2^-16), which covers its relative rounding at planes of 2^24
// columns.  NaN or infinite inputs fail every comparison.
constexpr float kOutsideBase = 131072.0f;   // 2^17
__device__ __forceinline__ bool window_outside(float cx, float cy, float cz, float h00, float h01,
                                               float h10, float h11, float h20, float h21, float R,
                                               float W, float H)
{
    constexpr float kE = 4.76837158203125e-07f;         // 2^-21
    constexpr float kOut = 1.0000152587890625f;         // 1 + 2^-16
    const float Wo = fmaf(W, kOut, 1.0f), Ho = fmaf(H, kOut, 1.0f);
    const float Tx = fmaf(R, fabsf(h00) + fabsf(h01), fabsf(cx));
    const float Ty = fmaf(R, fabsf(h10) + fabsf(h11), fabsf(cy));
    const float az = fabsf(h20) + fabsf(h21), Tz = fmaf(R, az, fabsf(cz));
    const float mx = kE * fmaf(Wo + kOutsideBase, Tz, Tx);
    const float my = kE * fmaf(Ho + kOutsideBase, Tz, Ty);
    // maxima of w_x + w_z and w_y + w_z; minima of w_x - Wo w_z, w_y - Ho w_z
    const float lx = fmaf(R, fabsf(h00 + h20) + fabsf(h01 + h21), cx + cz);
    const float ly = fmaf(R, fabsf(h10 + h20) + fabsf(h11 + h21), cy + cz);
    const float gx = fmaf(-R, fabsf(fmaf(-Wo, h20, h00)) + fabsf(fmaf(-Wo, h21, h01)),
                          fmaf(-Wo, cz, cx));
    const float gy = fmaf(-R, fabsf(fmaf(-Ho, h20, h10)) + fabsf(fmaf(-Ho, h21, h11)),
                          fmaf(-Ho, cz, cy));
    return fmaf(-kE, Tz, fmaf(-R, az, cz)) >= 1e-8f &&
           (lx + mx < 0.0f || ly + my < 0.0f || gx - mx > 0.0f || gy - my > 0.0f);
}

// True if every tap of the window has |w_z| >= 1e-8 in its FP32 evaluation:
// w_z is affine in the offset, so its extremes over |ox|, |oy| <= R are
// c_z -/+ R (|h20| + |h21|), each bound tightened by 2^-21 of the terms'
// magnitude as in window_inside (the taps' two FMAs, the bound's own
// rounding).  Then the masked loop's per-tap |w_z| test always passes.
__device__ __forceinline__ bool z_clear(float cz, float h20, float h21, float R)
{
    constexpr float kE = 4.76837158203125e-07f;   // 2^-21
    const float az = fabsf(h20) + fabsf(h21);
    const float Tz = fmaf(R, az, fabsf(cz));
    return (fmaf(-kE, Tz, fmaf(-R, az, cz)) >= 1e-8f) || (fmaf(kE, Tz, fmaf(R, az, cz)) <= -1e-8f);
}

}  // namespace hp3d
