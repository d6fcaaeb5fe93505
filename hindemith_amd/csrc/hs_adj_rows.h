// Fused reverse block of the Horn-Schunck adjoint for the canonical averaging
// stencil: one launch takes the state (u, v) m <= 8 steps before and the gradient
// after them, recomputes the m forward steps on chip and walks them backwards.
//
// What bounds it: vector issue, about 28 VALU instructions per cell and forward
// step, 22 per reverse step and 14 more on the tile's own rows, and, with one
// work-group per CU, the loads before the first step.  The two-launch form
// (hs_adj_tb_kernel after a recompute that stores each step's (ubar, vbar)) is
// bound by memory for large batches (64 B per pixel of them written and read again
// for 8 steps, besides 64 B of state, coefficients and accumulators; here they
// stay in registers) and by its tiles' latency for small ones.  Per 8 steps, two
// launches / this one: 3 x 243 x 331 31.9 / 18.6 us, 480x640 31.6 / 19.6, 8 x 512 x 512
// 112 / 100, 1920x1080 112 / 97; and the 2 planes per step are not allocated.
//
// Layout as hs_rows.h: a window of 64 columns x NW * P rows, a wave's P
// consecutive rows in registers, left and right neighbours through LDS, one
// barrier per step.  The steps are unrolled, so that each step's (ubar, vbar) has
// registers of its own; with P = 4 the first HL steps' go to LDS (their owner's
// cells only, so no barrier).
//
// Borders, forward: as hs_rows.h, except that the row below the image's last row
// is kept as a copy of it where it lies inside a strip (its owner copies it after
// each step).  Reverse: sources outside the image are zero (a cell of zeros for the
// columns, a row of zeros above and below), and a border pixel adds the gathers at
// its ghosts, of which only the terms with sources inside the image are left
// (hs_adj_tb_kernel's order).  Per-cell arithmetic and order are
// hs_adj_tb_kernel's: the same gradients.
#pragma once

#include <type_traits>

#include "hs_rows.h"

#pragma clang fp contract(off)

namespace hmx {

struct AdjRowsArgs {
    const float *Ix, *Iy, *It;
    const float *u, *v;          // the state m steps before
    const float *gu_in, *gv_in;  // the gradient after them
    float *gu_out, *gv_out;
    float *gIx, *gIy, *gIt, *ga2;  // accumulators (read unless first)
    const float *alpha2_b;
    int first;  // the accumulators start at zero
    int H, W, m, tw, th, tiles_x, ntiles;
    int64_t bstride;
    float w[8];
};

constexpr int ADJR_MMAX = 8;
constexpr int ADJR_COLS = HS_ROWS_COLS + 1;  // a window row and a cell of zeros

template <int NW, int P, int HL>
struct AdjRowsLds {
    float2 edge[2][NW][2][ADJR_COLS];
    float2 row[NW][P > 2 ? P - 2 : 1][ADJR_COLS];
    float2 zero[ADJR_COLS];
    float2 hist[HL ? HL : 1][HL ? NW : 1][HL ? P : 1][HL ? HS_ROWS_COLS : 1];
};

// 1/d rounded to nearest, from hs_recip where it accepts d
__device__ __forceinline__ float adj_recip_of(float r, float d) {
    if (r != r) {
        float dd = d;  // opaque: the division stays in the branch
        asm volatile("" : "+v"(dd));
        r = 1.0f / dd;
    }
    return r;
}

// Averaging weights held in vector registers, as kRowsVgprWeights; TWO builds: for two
// weights (hs_two_weights), where eight do not fit.
template <int P>
constexpr int kAdjVgprWeights = P == 2 ? 8 : 0;

template <int NW, int P, int HL, int WPE, bool TWO>
__global__ __launch_bounds__(64 * NW, WPE) void hs_adj_rows_kernel(AdjRowsArgs a) {
    static_assert(P >= 2 && P <= 4, "one group of rows per strip");
    __shared__ AdjRowsLds<NW, P, HL> lds;
    float w[8];
#pragma unroll
    for (int d = 0; d < 8; ++d)
        w[d] = TWO ? (d % 4 == 0 ? in_vgpr(a.w[d]) : w[d / 4 * 4])
                   : d < kAdjVgprWeights<P> ? in_vgpr(a.w[d]) : a.w[d];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int64_t off = (int64_t)blockIdx.y * a.bstride;
    const float alpha2 = a.alpha2_b[blockIdx.y];
    const int H = a.H, W = a.W, m = a.m;
    const int t = xcd_remap(blockIdx.x, a.ntiles);
    const int tyi = t / a.tiles_x, txi = t - tyi * a.tiles_x;
    const int x0 = txi * a.tw, y0 = tyi * a.th;
    const int x1 = min(x0 + a.tw, W), y1 = min(y0 + a.th, H);
    const int gx0 = x0 - m, gy0 = max(y0 - m, 0);
    const int gx = gx0 + lane;
    const int r0 = wave * P;
    const int jb = H - 1 - gy0 - r0;  // the image's last row, as a strip row
    const bool in = gx >= x0 && gx < x1;
    auto tile_row = [&](int j) { return gy0 + r0 + j >= y0 && gy0 + r0 + j < y1; };

    // byte offsets from the strip's first image row (uniform over the wave, 64 bits) fit
    // 32 bits; cells outside the image load the pixel they clamp to
    const int rs = min(gy0 + r0, H - 1);
    const int64_t strip = off + (int64_t)rs * W;
    const unsigned rowb = (unsigned)W * 4u;
    const unsigned co = (unsigned)clampi(gx, 0, W - 1) * 4u;
    auto at = [&](int j) { return (unsigned)(min(gy0 + r0 + j, H - 1) - rs) * rowb + co; };
    auto ld = [&](const float *plane, unsigned o) {
        return ld_g(reinterpret_cast<const float *>(
            reinterpret_cast<const char *>(plane + strip) + o));
    };
    float cx[P], cy[P], ct[P], cd[P], cr[P], u[P], v[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        u[j] = ld(a.u, at(j));
        v[j] = ld(a.v, at(j));
        cx[j] = ld(a.Ix, at(j));
        cy[j] = ld(a.Iy, at(j));
        ct[j] = ld(a.It, at(j));
    }
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const float m1 = cx[j] * cx[j];
        const float s1 = alpha2 + m1;
        const float m2 = cy[j] * cy[j];
        cd[j] = s1 + m2;
        cr[j] = hs_recip(cd[j]);
    }
    auto slot = [&](int buf, int j) -> float2 * {
        if (j == 0) return lds.edge[buf][wave][0];
        if (j == P - 1) return lds.edge[buf][wave][1];
        return lds.row[wave][j - 1];
    };
    auto wave_fence = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // forward neighbours: clamped to the image and the window
    const int lmin = max(-gx0, 0), lmax = min(W - 1 - gx0, HS_ROWS_COLS - 1);
    const int li = clampi(lane - 1, lmin, lmax), ri = clampi(lane + 1, lmin, lmax);
#pragma unroll
    for (int j = 0; j < P; ++j) slot(0, j)[lane] = make_float2(u[j], v[j]);
    // the zero cells and the zero row (first read after the reverse's first barrier)
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < P; ++j) slot(0, j)[ADJR_COLS - 1] = make_float2(0.0f, 0.0f);
        slot(1, 0)[ADJR_COLS - 1] = make_float2(0.0f, 0.0f);
        slot(1, P - 1)[ADJR_COLS - 1] = make_float2(0.0f, 0.0f);
        if (wave == 0) lds.zero[ADJR_COLS - 1] = make_float2(0.0f, 0.0f);
    }
    if (wave == 0) lds.zero[lane] = make_float2(0.0f, 0.0f);
    wave_fence();

    // (ubar, vbar) of forward step s = 0 .. m-1 at the thread's cells
    float2 hist[ADJR_MMAX - HL][P];
    // Forward step it (reads edge buffer (it - 1) & 1, writes the other), as hs_rows_tile.
    auto forward = [&](auto it_c) {
        constexpr int it = decltype(it_c)::value, buf = (it - 1) & 1;
        __syncthreads();
        const int lo = max(y0 - (m - it), 0) - gy0 - r0;
        const int hi = min(y1 + (m - it), H) - gy0 - r0;
        if (lo >= P || hi <= 0) return;
        const float2 *const ra =
            (gy0 + r0 == 0 || wave == 0) ? lds.edge[buf][wave][0] : lds.edge[buf][wave - 1][1];
        const float2 *const rb = (jb == P - 1 || wave == NW - 1) ? lds.edge[buf][wave][1]
                                                                 : lds.edge[buf][wave + 1][0];
        HsTri rows[P + 2];  // the old rows, one above and one below the strip
#pragma unroll
        for (int j = 0; j < P; ++j) {
            rows[j + 1].c = make_float2(u[j], v[j]);
            rows[j + 1].l = slot(buf, j)[li];
            rows[j + 1].r = slot(buf, j)[ri];
        }
        rows[0] = {ra[li], ra[lane], ra[ri]};
        rows[P + 1] = {rb[li], rb[lane], rb[ri]};
        float ub[P], vb[P], s2[P], q[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const HsTri &up = rows[j], &me = rows[j + 1], &dn = rows[j + 2];
            float x = 0.0f, y = 0.0f;
            auto tap = [&](int d, float2 z) {
                x = fmaf(w[d], z.x, x);
                y = fmaf(w[d], z.y, y);
            };
            tap(0, me.l);  // HS_RING_OX/OY order
            tap(1, me.r);
            tap(2, up.c);
            tap(3, dn.c);
            tap(4, up.l);
            tap(5, up.r);
            tap(6, dn.l);
            tap(7, dn.r);
            ub[j] = x;
            vb[j] = y;
            const float m1 = cx[j] * x;
            const float m2 = cy[j] * y;
            const float s1 = m1 + m2;
            s2[j] = s1 + ct[j];
            q[j] = hs_quotient(s2[j], cd[j], cr[j]);
        }
        float mx = fabsf(q[0]), mn = mx;
#pragma unroll
        for (int j = 1; j < P; ++j) {
            mx = __builtin_elementwise_maximum(mx, fabsf(q[j]));
            mn = __builtin_elementwise_minimum(mn, fabsf(q[j]));
        }
        if (!(mn >= 0x1p-76f && mx <= 0x1p76f)) {
#pragma unroll
            for (int j = 0; j < P; ++j) {
                float so = s2[j];
                asm volatile("" : "+v"(so));
                q[j] = so / cd[j];
            }
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const float p1 = cx[j] * q[j];
            const float p2 = cy[j] * q[j];
            u[j] = ub[j] - p1;
            v[j] = vb[j] - p2;
            if constexpr (it - 1 < HL)
                lds.hist[it - 1][wave][j][lane] = make_float2(ub[j], vb[j]);
            else
                hist[it - 1 - HL][j] = make_float2(ub[j], vb[j]);
        }
        // the row below the image's last row
        if (jb >= 0 && jb < P - 1) {
#pragma unroll
            for (int j = 0; j + 1 < P; ++j)
                if (j == jb) {
                    u[j + 1] = u[j];
                    v[j + 1] = v[j];
                }
        }
#pragma unroll
        for (int j = 0; j < P; ++j) slot(buf ^ 1, j)[lane] = make_float2(u[j], v[j]);
        wave_fence();
    };
    // (the last step's new state is not needed, but its (ubar, vbar) are)
    auto each_step = [](auto &&f) {
        f(std::integral_constant<int, 1>());
        f(std::integral_constant<int, 2>());
        f(std::integral_constant<int, 3>());
        f(std::integral_constant<int, 4>());
        f(std::integral_constant<int, 5>());
        f(std::integral_constant<int, 6>());
        f(std::integral_constant<int, 7>());
        f(std::integral_constant<int, 8>());
    };
    float2 g[P];
    float ax[P], ay[P], az[P], aa[P];
    // the gradient and the accumulators: their reads are covered by the forward steps
#pragma unroll
    for (int j = 0; j < P; ++j) {
        g[j] = make_float2(ld(a.gu_in, at(j)), ld(a.gv_in, at(j)));
        ax[j] = ay[j] = az[j] = aa[j] = 0.0f;
        if (!a.first && tile_row(j) && in) {
            ax[j] = ld(a.gIx, at(j));
            ay[j] = ld(a.gIy, at(j));
            az[j] = ld(a.gIt, at(j));
            aa[j] = ld(a.ga2, at(j));
        }
    }
    each_step([&](auto it_c) {
        if (decltype(it_c)::value <= m) forward(it_c);
    });

    // ---- reverse ----
    // neighbours: the zero cell beyond the image's first and last columns
    const int zl = gx == 0 ? ADJR_COLS - 1 : max(lane - 1, 0);
    const int zr = gx == W - 1 ? ADJR_COLS - 1 : min(lane + 1, HS_ROWS_COLS - 1);
    // the strip holds border pixels, or rows below the image (uniform: most strips
    // gather without the border terms and their branches)
    const bool border =
        gx0 <= 0 || gx0 + HS_ROWS_COLS >= W || gy0 + r0 == 0 || jb < P;
    float2 G[P];  // (g_ubar, g_vbar)
#pragma unroll
    for (int j = 0; j < P; ++j) cr[j] = adj_recip_of(cr[j], cd[j]);
    // pass A at strip row j: s and (g_ubar, g_vbar)
    float sv[P];
    auto pass_a = [&](int j) {
        sv[j] = -fmaf(cx[j], g[j].x, cy[j] * g[j].y) * cr[j];
        G[j] = make_float2(fmaf(cx[j], sv[j], g[j].x), fmaf(cy[j], sv[j], g[j].y));
    };
    // and the accumulators' terms, about the forward step that lin belongs to (for
    // every row of a strip that has tile rows: the others are not stored)
    auto accumulate = [&](int j, float2 lin) {
        const float s = sv[j];
        const float tt = (fmaf(cx[j], lin.x, cy[j] * lin.y) + ct[j]) * cr[j];
        const float st2 = 2.0f * s * tt;
        ax[j] = fmaf(-st2, cx[j], fmaf(s, lin.x, fmaf(-g[j].x, tt, ax[j])));
        ay[j] = fmaf(-st2, cy[j], fmaf(s, lin.y, fmaf(-g[j].y, tt, ay[j])));
        az[j] += s;
        aa[j] = fmaf(-s, tt, aa[j]);
    };
    const bool tiled = gy0 + r0 < y1 && gy0 + r0 + P > y0;
    // rows below the image stay zero
    auto below_zero = [&]() {
#pragma unroll
        for (int j = 1; j < P; ++j)
            if (j > jb) G[j] = make_float2(0.0f, 0.0f);
        if (jb < 0) G[0] = make_float2(0.0f, 0.0f);
    };
    auto lin_of = [&](auto f_c, int j) -> float2 {
        constexpr int f = decltype(f_c)::value;  // forward step index
        if constexpr (f < HL)
            return lds.hist[f][wave][j][lane];
        else
            return hist[f - HL][j];
    };
    // the forward's last step was m: start with pass A about step m - 1 on every
    // row of the window
    auto start = [&](auto f_c) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
            pass_a(j);
            accumulate(j, lin_of(f_c, j));
        }
        below_zero();
    };
    __syncthreads();  // every wave is past its last read of the forward's edge rows
    switch (m) {
        case 1: start(std::integral_constant<int, 0>()); break;
        case 2: start(std::integral_constant<int, 1>()); break;
        case 3: start(std::integral_constant<int, 2>()); break;
        case 4: start(std::integral_constant<int, 3>()); break;
        case 5: start(std::integral_constant<int, 4>()); break;
        case 6: start(std::integral_constant<int, 5>()); break;
        case 7: start(std::integral_constant<int, 6>()); break;
        default: start(std::integral_constant<int, 7>()); break;
    }
    // pass B then pass A: reverse step s walks back over forward step m - s.  F = m - s
    // is the compile-time index here: steps F = 7 .. 0, those with F < m.  Step F
    // reads edge buffer F & 1 and writes the other.
#pragma unroll
    for (int j = 0; j < P; ++j) {
        slot(0, j)[lane] = G[j];
        if (j == 0 || j == P - 1) slot(1, j)[lane] = G[j];
    }
    wave_fence();
    auto backward = [&](auto f_c) {
        constexpr int F = decltype(f_c)::value, buf = F & 1;
        __syncthreads();
        // rows of reach F: the tile grown by F
        const int lo = max(y0 - F, 0) - gy0 - r0;
        const int hi = min(y1 + F, H) - gy0 - r0;
        if (lo >= P || hi <= 0) return;
        const float2 *const ra = gy0 + r0 == 0 ? lds.zero
                                 : wave == 0   ? lds.edge[buf][wave][0]
                                               : lds.edge[buf][wave - 1][1];
        const float2 *const rb = jb == P - 1       ? lds.zero
                                 : wave == NW - 1 ? lds.edge[buf][wave][1]
                                                  : lds.edge[buf][wave + 1][0];
        HsTri rows[P + 2];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            rows[j + 1].c = G[j];
            rows[j + 1].l = slot(buf, j)[zl];
            rows[j + 1].r = slot(buf, j)[zr];
        }
        rows[0] = {ra[zl], ra[lane], ra[zr]};
        rows[P + 1] = {rb[zl], rb[lane], rb[zr]};
        // BORDER: the strip holds border pixels or rows below the image
        auto gather = [&](auto border_c) {
            constexpr bool BORDER = decltype(border_c)::value;
#pragma unroll
            for (int j = 0; j < P; ++j) {
                if (BORDER && j > jb) continue;  // below the image: stays zero
                const HsTri &up = rows[j], &me = rows[j + 1], &dn = rows[j + 2];
                float x = 0.0f, y = 0.0f;
                auto tap = [&](int d, float2 z) {
                    x = fmaf(w[d], z.x, x);
                    y = fmaf(w[d], z.y, y);
                };
                tap(0, me.r);  // the source of tap d lies at -(ox, oy)
                tap(1, me.l);
                tap(2, dn.c);
                tap(3, up.c);
                tap(4, dn.r);
                tap(5, dn.l);
                tap(6, up.r);
                tap(7, up.l);
                if (BORDER) {
                    // border pixels: the gathers at their ghosts
                    const bool bl = gx == 0, br = gx == W - 1;
                    if (bl) {
                        tap(0, me.c);
                        tap(4, dn.c);
                        tap(6, up.c);
                    }
                    if (br) {
                        tap(1, me.c);
                        tap(5, dn.c);
                        tap(7, up.c);
                    }
                    if (j == 0 && gy0 + r0 == 0) {
                        tap(2, me.c);
                        tap(4, me.r);
                        tap(5, me.l);
                        if (bl) tap(4, me.c);
                        if (br) tap(5, me.c);
                    }
                    if (j == jb) {
                        tap(3, me.c);
                        tap(6, me.r);
                        tap(7, me.l);
                        if (bl) tap(6, me.c);
                        if (br) tap(7, me.c);
                    }
                }
                g[j] = make_float2(x, y);
            }
        };
        if (border)
            gather(std::true_type());
        else
            gather(std::false_type());
        if constexpr (F > 0) {
#pragma unroll
            for (int j = 0; j < P; ++j) pass_a(j);
            if (tiled) {
#pragma unroll
                for (int j = 0; j < P; ++j)
                    accumulate(j, lin_of(std::integral_constant<int, F - 1>(), j));
            }
            if (jb < P - 1) below_zero();
#pragma unroll
            for (int j = 0; j < P; ++j) slot(buf ^ 1, j)[lane] = G[j];
            wave_fence();
        }
    };
    if (m > 7) backward(std::integral_constant<int, 7>());
    if (m > 6) backward(std::integral_constant<int, 6>());
    if (m > 5) backward(std::integral_constant<int, 5>());
    if (m > 4) backward(std::integral_constant<int, 4>());
    if (m > 3) backward(std::integral_constant<int, 3>());
    if (m > 2) backward(std::integral_constant<int, 2>());
    if (m > 1) backward(std::integral_constant<int, 1>());
    backward(std::integral_constant<int, 0>());

    if (in) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
            if (!tile_row(j)) continue;
            const unsigned o = at(j);
            auto st = [&](float *plane, float x) {
                *(gfloat *)(reinterpret_cast<char *>(plane + strip) + o) = x;
            };
            st(a.gu_out, g[j].x);
            st(a.gv_out, g[j].y);
            st(a.gIx, ax[j]);
            st(a.gIy, ay[j]);
            st(a.gIt, az[j]);
            st(a.ga2, aa[j]);
        }
    }
}

}  // namespace hmx
