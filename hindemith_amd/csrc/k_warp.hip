// a17: WarpImg2D -- bilinear warp of an image by a per-pixel offset field
// (WarpImg2D.cpp:33-75), the building block of coarse-to-fine / warped HS.
//
// dst(x, y) = bilinear sample of src at (x + offx, y + offy) when all four
// taps lie inside the image, else src(x, y).  The offset splits into an
// integer part by truncation, moved down by one for negative offsets (so the
// fraction lies in [0, 1]).
//
// The generated code mixes float data with double literals (1.0); this
// kernel evaluates each statement in the type C gives it: the weights
// 1.0 - frac in double, float products where both operands are float, and
// each "out += term" as one fma in the statement's type, rounded to float on
// assignment -- the same convention as the other accumulations here.
#include "hmx_common.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace hmx {

// A pixel's sample: the element offset of its upper left tap and the fractions, or
// (inside false) none: the pixel's own value.
struct WarpSample {
    int64_t q;
    float xf, yf;
    bool inside;
};

__device__ __forceinline__ WarpSample warp_sample(float ox, float oy, int r, int c, int H, int W) {
    WarpSample s;
    int mx = (int)ox, my = (int)oy;
    s.xf = ox - (float)mx;
    s.yf = oy - (float)my;
    if (ox < 0.0f) {
        --mx;
        s.xf = (float)(1.0 + (double)s.xf);
    }
    if (oy < 0.0f) {
        --my;
        s.yf = (float)(1.0 + (double)s.yf);
    }
    const int64_t sx = (int64_t)c + mx, sy = (int64_t)r + my;
    s.inside = sx >= 0 && sx + 1 < W && sy >= 0 && sy + 1 < H;
    s.q = sy * W + sx;
    return s;
}

__device__ __forceinline__ float warp_blend(const WarpSample &s, float i00, float i10, float i01,
                                            float i11) {
    const double ax = 1.0 - (double)s.xf, ay = 1.0 - (double)s.yf;
    float out = 0.0f;
    out = (float)fma((double)i00 * ax, ay, (double)out);            // IN00*(1-xf)*(1-yf)
    const float p10 = i10 * s.xf;
    out = (float)fma((double)p10, ay, (double)out);                 // IN10*xf*(1-yf)
    out = (float)fma((double)i01 * ax, (double)s.yf, (double)out);  // IN01*(1-xf)*yf
    const float p11 = i11 * s.xf;
    out = fmaf(p11, s.yf, out);                                     // IN11*xf*yf
    return out;
}

// 16 B/px: read offx, offy and (once, through the cache) src; write dst.  V rows of
// a column per thread: all their offsets are read before the first tap and all taps
// before the first blend.  (The value of a pixel whose taps are outside has a register
// of its own: sharing a tap's would make the wave wait for one branch's load before
// it issues the other's.)
template <int V>
__global__ __launch_bounds__(256) void warp_img2d_kernel(const float *__restrict__ src,
                                                         const float *__restrict__ offx,
                                                         const float *__restrict__ offy,
                                                         float *__restrict__ dst, int H, int W) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= W) return;
    const bool wt = rows_whole_lines(W);
    for (int r0 = blockIdx.y * V; r0 < H; r0 += gridDim.y * V) {
        float ox[V], oy[V], t[V][4], own[V];
        WarpSample s[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int64_t p = (int64_t)min(r0 + v, H - 1) * W + c;
            ox[v] = offx[p];
            oy[v] = offy[p];
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            s[v] = warp_sample(ox[v], oy[v], min(r0 + v, H - 1), c, H, W);
            const float *const a = src + (s[v].inside ? s[v].q : 0);
            if (s[v].inside) {
                t[v][0] = a[0];
                t[v][1] = a[1];
                t[v][2] = a[W];
                t[v][3] = a[W + 1];
            } else {
                own[v] = src[(int64_t)min(r0 + v, H - 1) * W + c];
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (r0 + v < H)
                st_out(dst + (int64_t)(r0 + v) * W + c,
                       s[v].inside ? warp_blend(s[v], t[v][0], t[v][1], t[v][2], t[v][3]) : own[v],
                       wt);
    }
}

int launch_warp_img2d(const float *src, const float *offx, const float *offy, float *dst, int H,
                      int W, hipStream_t s) {
    // A pixel's taps wait for its offsets, two memory latencies one after the other.
    // From about a megapixel that wait is the bound, and four pixels per thread keep
    // four times the reads in flight (us, one pixel / four: 3840x2160 40 / 26.7, 5.0
    // TB/s; 2560x1440 19.4 / 15; 1920x1080 10.3 / 8.6); below it more work-groups are
    // worth more (977x613 3.6 / 4.5, 240x135 2.2 / 2.7).  Offsets that are random by tens
    // of pixels from each pixel to the next are bound by their lines, and lose up to 9 %
    // below 2.5 Mpixel (1920x1080 19.3 / 20.4).
    const bool large = (int64_t)H * W >= (int64_t)1 << 20;
    const int v = large ? 4 : 1;
    dim3 grid((W + 255) / 256, std::min((H + v - 1) / v, 65535));
    if (large)
        hipLaunchKernelGGL(warp_img2d_kernel<4>, grid, dim3(256), 0, s, src, offx, offy, dst, H, W);
    else
        hipLaunchKernelGGL(warp_img2d_kernel<1>, grid, dim3(256), 0, s, src, offx, offy, dst, H, W);
    HMX_LAUNCH_CHECK("warp_img2d");
    return HMX_OK;
}

}  // namespace hmx

using namespace hmx;

extern "C" int hmx_warp_img2d(const float *src, const float *offx, const float *offy, float *dst,
                              int H, int W, void *stream) {
    HMX_REQUIRE(src && offx && offy && dst, "hmx_warp_img2d: null argument");
    HMX_REQUIRE(H > 0 && W > 0, "hmx_warp_img2d: H and W must be positive");
    HMX_REQUIRE(dst != src && dst != offx && dst != offy,
                "hmx_warp_img2d: dst must be distinct from the inputs");
    return launch_warp_img2d(src, offx, offy, dst, H, W, as_stream(stream));
}
