// Operations of the reference's preconditioned-CG Horn-Schunck solver:
//   a15  ApplyHSPreconditioner  (ApplyHSPreconditioner.cpp:46-97)
//   a16  HSMatrixPowers         (HSMatrixPowers.cpp:28-39, 72-126, 191-226)
//
// The HS normal-equation operator on x = (u, v), with I = (Ix, Iy) and L the
// 4-neighbour Laplacian with Neumann (no-flux) borders weighted by lambda:
//   A x = ( Ix (Ix u + Iy v) + lam L u ,  Iy (Ix u + Iy v) + lam L v ).
// Its per-pixel 2x2 diagonal block [[a, b], [b, d]] with a = diag0 + n_nb*w2,
// d = diag1 + n_nb*w2 (n_nb = in-image 4-neighbours, w2 = weight 2 of the
// stencil passed in) is what the preconditioner inverts.
//
// Arithmetic follows the generated OpenCL statement by statement: one
// rounding per operator, the "y += p * q" accumulations of HSMatrixPowers as
// fmas (as the stencil accumulation elsewhere), correctly rounded division.
#include "hmx_common.h"
#include "hs_rows.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace hmx {

// ---------------------------------------------------------------------------
// a15: y = M^-1 x per pixel.  28 B/px (read diag0, diag1, offdiag, x0, x1;
// write y0, y1): HBM bound, one pixel per thread, row-major order.
__global__ __launch_bounds__(256) void hs_precond_kernel(
    const float *__restrict__ diag0, const float *__restrict__ diag1,
    const float *__restrict__ offdiag, const float *__restrict__ x0,
    const float *__restrict__ x1, float *__restrict__ y0, float *__restrict__ y1, int H, int W,
    const float *__restrict__ w_dev, float w_val) {
    const int64_t n = (int64_t)H * W;
    const float s2 = w_dev ? w_dev[2] : w_val;  // the stencil's weight 2 (getData("2"))
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
         p += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(p / W), c = (int)(p - (int64_t)r * W);
        float a = diag0[p], d = diag1[p];
        // neighbour terms in the order of the generated code
        if (c < W - 1) { a = a + s2; d = d + s2; }
        if (r < H - 1) { a = a + s2; d = d + s2; }
        if (c > 0) { a = a + s2; d = d + s2; }
        if (r > 0) { a = a + s2; d = d + s2; }
        const float b = offdiag[p];
        const float e = x0[p], f = x1[p];
        const float ad = a * d, bc = b * b;
        const float det = ad - bc;
        // 1e-15 is a double literal in the generated code: compare in double
        if (fabs((double)det) > 1e-15) {
            const float t0 = e * d, t1 = b * f;
            const float n0 = t0 - t1;
            const float t2 = (-b) * e, t3 = a * f;
            const float n1 = t2 + t3;
            y0[p] = n0 / det;
            y1[p] = n1 / det;
        } else {
            st_out(y0 + p, e, true);
            st_out(y1 + p, f, true);
        }
    }
}

// ---------------------------------------------------------------------------
// a16: V[0] = r, V[s] = A V[s-1] for s = 1..steps-1, all powers stored.
//
// Temporally blocked like the Jacobi sweep, in its row-register layout
// (hs_rows_tile): a work-group loads r, Ix and Iy on its tile grown by m =
// (powers this launch) pixels and computes the m powers on chip; power j is valid
// on the tile grown by m - j.  A lane is a window column, a wave owns POW_P
// window rows in registers, and only left and right neighbours (a wave's own
// rows) and the rows where two waves meet go through LDS: 3 LDS operations per
// cell and power, one barrier per power.  Each power's tile is stored as it is
// made, so HBM traffic per launch is 16 B/px read + 8 B/px per power written (the
// per-power launches of the reference move 24 B/px per power).
//
// What bounds it: the stores.  8 powers and r of 3840x2160 are 597 MB out and 133 MB
// in, 119 us at the rates of a fill (6.9 TB/s) and a read (4.2); without its stores
// the kernel takes 100 us.  Measured, 8 powers: 3840x2160 161 us (a 64x32 tile with
// every cell's neighbours read from LDS: 239, 183 with non-temporal stores),
// 1920x1080 35 (43.5), 135x240 11 (13.7).  Tiles are POW_TW = 48 columns, three
// 64-byte sectors a row: 32-column tiles in whole cache lines cost 214 us in redundant
// columns; windows of 48 to 96 rows and 8 to 16 waves lie within 155 - 177.
constexpr int POW_MMAX = 8, POW_TW = HS_ROWS_COLS - 2 * POW_MMAX;
constexpr int POW_NW = 16, POW_P = 4;  // waves, window rows per wave

struct PowArgs {
    const float *Ix, *Iy;
    const float *u0, *v0;  // power s0 - 1 (V[0] = r on the first launch)
    float *V0, *V1;        // steps x H x W
    int s0, m;             // this launch makes powers s0 .. s0+m-1
    int H, W, th, tiles_x, ntiles;
    int64_t plane;         // H * W
    const void *lam_dev;   // device scalar of dtype lam_dtype, or null: lam_val
    int lam_dtype;
    float lam_val;
    int copy_r;            // also store V[0] = r (the Array2D -> Array3D copy)
};

template <int NW, int P, bool NTS>
__global__ __launch_bounds__(NW * 64, 8) void hs_powers_kernel(PowArgs a) {
    __shared__ HsRowsLds<NW, P> lds;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int H = a.H, W = a.W, m = a.m;
    const int t = xcd_remap(blockIdx.x, a.ntiles);
    const int tyi = t / a.tiles_x, txi = t - tyi * a.tiles_x;
    const int x0 = txi * POW_TW, y0 = tyi * a.th;
    const int x1 = min(x0 + POW_TW, W), y1 = min(y0 + a.th, H);
    // window: columns x0 - m .., rows from y0 - m, or from the image's first
    const int gx0 = x0 - m, gy0 = max(y0 - m, 0);
    const int gx = gx0 + lane;
    const int r0 = wave * P;  // the strip's first window row
    // a row's address is uniform over its wave (64-bit offsets, for planes of any
    // size); a lane adds its column's distance from the window's first
    const unsigned co = (unsigned)(clampi(gx, 0, W - 1) - gx0) * 4u;
    const unsigned lane4 = (unsigned)lane * 4u;
    float cx[P], cy[P], u[P], v[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int64_t o = (int64_t)min(gy0 + r0 + j, H - 1) * W + gx0;
        auto ld = [&](const float *p) {
            return ld_g(reinterpret_cast<const float *>(reinterpret_cast<const char *>(p + o) + co));
        };
        u[j] = ld(a.u0);
        v[j] = ld(a.v0);
        cx[j] = ld(a.Ix);
        cy[j] = ld(a.Iy);
    }
    // a scalar of another dtype is rounded to float32 first
    float lam = a.lam_val;
    if (a.lam_dev) {
        switch (a.lam_dtype) {
            case HMX_F64: lam = (float)*(const double *)a.lam_dev; break;
            case HMX_I64: lam = (float)*(const long long *)a.lam_dev; break;
            case HMX_I32: lam = (float)*(const int *)a.lam_dev; break;
            default: lam = *(const float *)a.lam_dev; break;
        }
    }
    const float nlam = -lam;
    const int li = max(lane - 1, 0), ri = min(lane + 1, HS_ROWS_COLS - 1);
    const bool in = gx >= x0 && gx < x1;
    const bool has_l = gx > 0, has_r = gx < W - 1;
    // the strip's rows in the output tile
    unsigned tile_rows = 0;
    for (int j = 0; j < P; ++j)
        if (gy0 + r0 + j >= y0 && gy0 + r0 + j < y1) tile_rows |= 1u << j;
    // rows of power s: uniform row addresses plus the lane's offset (opaque, so that
    // it is added by the store and not before, in 64-bit vector additions)
    auto store = [&](int s, const float (&p)[P], const float (&q)[P]) {
        const int64_t o = (int64_t)s * a.plane + (int64_t)(gy0 + r0) * W + gx0;
        float *row0 = a.V0 + o, *row1 = a.V1 + o;
#pragma unroll
        for (int j = 0; j < P; ++j, row0 += W, row1 += W) {
            if (!((tile_rows >> j) & 1)) continue;
            auto st = [&](float *row, float x) {
                unsigned l4 = lane4;
                asm volatile("" : "+v"(l4));
                gfloat *const g = (gfloat *)(reinterpret_cast<char *>(row) + l4);
                if (NTS)
                    __builtin_nontemporal_store(x, g);
                else
                    *g = x;
            };
            st(row0, p[j]);
            st(row1, q[j]);
        }
    };
    if (a.copy_r && in) store(0, u, v);
    auto slot = [&](int buf, int j) -> float2 * {
        if (j == 0) return lds.edge[buf][wave][0];
        if (j == P - 1) return lds.edge[buf][wave][1];
        return lds.row[wave][j - 1];
    };
    // a wave's LDS writes before its reads of the same row (a wavefront's LDS
    // accesses are performed in order; this keeps the compiler's order)
    auto wave_fence = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
#pragma unroll
    for (int j = 0; j < P; ++j) slot(0, j)[lane] = make_float2(u[j], v[j]);
    wave_fence();

    auto steps = [&](auto clip_c) {
        constexpr bool CLIP = decltype(clip_c)::value;
        for (int it = 1; it <= m; ++it) {
            // power it reads edge buffer (it - 1) & 1 and writes the other, which was
            // last read for power it - 1, before this barrier
            __syncthreads();
            const int buf = (it - 1) & 1;
            // active strip rows [lo, hi): the tile grown by m - it, inside the image
            const int lo = max(y0 - (m - it), 0) - gy0 - r0;
            const int hi = min(y1 + (m - it), H) - gy0 - r0;
            if (lo >= P || hi <= 0) continue;
            const float2 *const ra =
                wave == 0 ? lds.edge[buf][wave][0] : lds.edge[buf][wave - 1][1];
            const float2 *const rb =
                wave == NW - 1 ? lds.edge[buf][wave][1] : lds.edge[buf][wave + 1][0];
            const float2 above = ra[lane], below = rb[lane];
            float nu[P], nv[P];
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const float2 l = slot(buf, j)[li], r = slot(buf, j)[ri];
                const float2 up = j == 0 ? above : make_float2(u[j > 0 ? j - 1 : 0],
                                                               v[j > 0 ? j - 1 : 0]);
                const float2 dn = j == P - 1 ? below : make_float2(u[j < P - 1 ? j + 1 : j],
                                                                   v[j < P - 1 ? j + 1 : j]);
                const float p1 = cx[j] * u[j], p2 = cy[j] * v[j];
                const float dot = p1 + p2;
                float x = cx[j] * dot, y = cy[j] * dot;
                auto nb = [&](float2 q, bool has) {
                    float xn = fmaf(nlam, q.x, x), yn = fmaf(nlam, q.y, y);
                    xn = fmaf(lam, u[j], xn);
                    yn = fmaf(lam, v[j], yn);
                    x = !CLIP || has ? xn : x;
                    y = !CLIP || has ? yn : y;
                };
                const int gy = gy0 + r0 + j;
                nb(l, has_l);
                nb(r, has_r);
                nb(up, gy > 0);
                nb(dn, gy < H - 1);
                nu[j] = x;
                nv[j] = y;
            }
#pragma unroll
            for (int j = 0; j < P; ++j) {
                u[j] = nu[j];
                v[j] = nv[j];
                slot(buf ^ 1, j)[lane] = make_float2(nu[j], nv[j]);
            }
            if (in) store(a.s0 + it - 1, u, v);
            wave_fence();
        }
    };
    if (gx0 <= 0 || y0 - m <= 0 || x1 + m >= W || y1 + m >= H)
        steps(std::true_type());
    else
        steps(std::false_type());
}

int launch_hs_precond(const float *diag0, const float *diag1, const float *offdiag,
                      const float *x0, const float *x1, float *y0, float *y1, int H, int W,
                      const float *w_dev, float w_val, hipStream_t s) {
    const int64_t n = (int64_t)H * W;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 1 << 20);
    hipLaunchKernelGGL(hs_precond_kernel, dim3((unsigned)blocks), dim3(256), 0, s, diag0, diag1,
                       offdiag, x0, x1, y0, y1, H, W, w_dev, w_val);
    HMX_LAUNCH_CHECK("hs_precond");
    return HMX_OK;
}

// V0, V1: steps planes of H x W.  Powers are made POW_MMAX per launch; each
// launch after the first starts from the last power the previous one stored.
int launch_hs_powers(const float *Ix, const float *Iy, const float *r0, const float *r1,
                     float *V0, float *V1, int H, int W, int steps, const void *lam_dev,
                     int lam_dtype, float lam_val, hipStream_t s) {
    PowArgs a;
    a.Ix = Ix;
    a.Iy = Iy;
    a.V0 = V0;
    a.V1 = V1;
    a.H = H;
    a.W = W;
    a.plane = (int64_t)H * W;
    a.tiles_x = (W + POW_TW - 1) / POW_TW;
    a.lam_dev = lam_dev;
    a.lam_dtype = lam_dtype;
    a.lam_val = lam_val;
    if (steps == 1) {  // only V[0] = r
        HMX_HIP_TRY(hipMemcpyAsync(V0, r0, a.plane * 4, hipMemcpyDeviceToDevice, s));
        HMX_HIP_TRY(hipMemcpyAsync(V1, r1, a.plane * 4, hipMemcpyDeviceToDevice, s));
        return HMX_OK;
    }
    // Non-temporal stores pay where the powers outgrow the 256 MB memory-side cache
    // anyway and a row starts on a 64-byte sector, so that a tile row's 192 bytes are
    // whole ones.  us for 8 powers, plain / non-temporal: 3840x2160 205 / 155, 2560x1440
    // (265 MB) 94 / 71, 1920x1080 (149 MB) 37 / 35; 2100x1200, rows off the sectors, 44
    // / 87; smaller ones alike, and a consumer then finds plain ones cached.
    const bool nts = (W & 15) == 0 && 2 * (int64_t)steps * a.plane * 4 >= ((int64_t)128 << 20);
    for (int s0 = 1; s0 < steps; s0 += POW_MMAX) {
        a.s0 = s0;
        a.m = std::min(POW_MMAX, steps - s0);
        a.th = POW_NW * POW_P - 2 * a.m;
        a.ntiles = a.tiles_x * ((H + a.th - 1) / a.th);
        a.copy_r = s0 == 1;
        a.u0 = s0 == 1 ? r0 : V0 + (int64_t)(s0 - 1) * a.plane;
        a.v0 = s0 == 1 ? r1 : V1 + (int64_t)(s0 - 1) * a.plane;
        if (nts)
            hipLaunchKernelGGL((hs_powers_kernel<POW_NW, POW_P, true>), dim3(a.ntiles),
                               dim3(POW_NW * 64), 0, s, a);
        else
            hipLaunchKernelGGL((hs_powers_kernel<POW_NW, POW_P, false>), dim3(a.ntiles),
                               dim3(POW_NW * 64), 0, s, a);
        HMX_LAUNCH_CHECK("hs_powers");
    }
    return HMX_OK;
}

}  // namespace hmx

using namespace hmx;

extern "C" int hmx_hs_precondition(const float *diag0, const float *diag1, const float *offdiag,
                                   const float *x0, const float *x1, float *y0, float *y1,
                                   int H, int W, int nd, const float *w, void *stream) {
    HMX_REQUIRE(diag0 && diag1 && offdiag && x0 && x1 && y0 && y1 && w,
                "hmx_hs_precondition: null argument");
    HMX_REQUIRE(H > 0 && W > 0, "hmx_hs_precondition: H and W must be positive");
    HMX_REQUIRE(nd >= 3, "hmx_hs_precondition: the stencil needs a weight 2 (>= 3 taps)");
    HMX_REQUIRE(y0 != x0 && y0 != x1 && y1 != x0 && y1 != x1 && y0 != y1,
                "hmx_hs_precondition: outputs must be distinct from the inputs");
    return launch_hs_precond(diag0, diag1, offdiag, x0, x1, y0, y1, H, W, nullptr, w[2],
                             as_stream(stream));
}

extern "C" int hmx_hs_matrix_powers(float lam, const float *Ix, const float *Iy,
                                    const float *r0, const float *r1, float *V0, float *V1,
                                    int H, int W, int steps, void *stream) {
    HMX_REQUIRE(Ix && Iy && r0 && r1 && V0 && V1, "hmx_hs_matrix_powers: null argument");
    HMX_REQUIRE(H > 0 && W > 0, "hmx_hs_matrix_powers: H and W must be positive");
    HMX_REQUIRE(steps >= 1, "hmx_hs_matrix_powers: steps must be >= 1");
    HMX_REQUIRE(H < 32768 && W < 32768, "hmx_hs_matrix_powers: H and W must be < 32768");
    return launch_hs_powers(Ix, Iy, r0, r1, V0, V1, H, W, steps, nullptr, HMX_F32, lam,
                            as_stream(stream));
}
