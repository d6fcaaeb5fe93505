// Row-register tile body of the fused Horn-Schunck Jacobi sweep for the
// canonical 8-tap averaging stencil (hs_ring_taps).
//
// Like hs_tile, a work-group advances one output tile by k steps on chip: the
// window is the tile grown by k pixels, and step `it` updates the tile grown
// by k - it.  Here the window is 64 columns wide, one lane per column, and
// wave q of the work-group owns P consecutive window rows: a thread keeps (u, v)
// and the coefficients of its P cells of one column in registers.  A cell's
// upper and lower neighbours are then the thread's own registers; only the
// left and right ones go through LDS, and those are a wave's own rows, so a
// step has one barrier, for the rows where two waves meet.
//
// What bounds it: vector issue, and, where a CU holds one or two tiles, the loads
// before the first step.  hs_tile reads 8 neighbours per cell from LDS
// (9 LDS operations of 4 cycles per wave-cell against 33 VALU instructions: the
// two units are equally loaded and neither hides the other's latency); this
// body does 3 LDS operations and 29 VALU instructions per cell, no activity
// test (a wave's strip is active in its first steps and not after them) and no
// address arithmetic (every LDS access is one of three registers plus a constant), and its prologue takes ~20 instructions per cell instead of ~47.
// Its operands are vector registers (in_vgpr), which two waves issue together.
// Measured, us per 8 iterations, hs_tile's variant 24 / this body with scalar
// weights, two corrections per quotient and a branch per row / as it is: 135x240
// 12.5 / 5.8 / 5.1, 480x640 12.9 / 9.1 / 7.8, 613x977 19.4 / 12.3 / 10.8, 1920x1080
// 33.6 / 32.3 / 26.7, 3840x2160 112 / 98 / 90.
//
// Replicated borders cost nothing per step: the lane a cell takes its left (right)
// neighbour from is clamped to the image once per tile, a window never starts
// above the image, and the row below the image's last row is that row itself
// (its wave selects it; if it is the strip's last row, by the address it reads).
// Cells outside the image load the pixel they clamp to and are never read by
// an image cell.
//
// The arithmetic is hs_update's, in the same order, so results are bit-identical
// to every other variant: averages as fma chains in tap order from 0, the
// quotient from the per-cell reciprocal (hs_div.h).  Its range check is made once
// for a group of up to G cells (|q| of all of them through one minimum and one maximum
// chain, NaN propagating); a lane that fails it divides all of them.
#pragma once

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "hmx_common.h"
#include "hs_div.h"
#include "hs_tile.h"

#pragma clang fp contract(off)

namespace hmx {

constexpr int HS_ROWS_COLS = 64;  // window columns: one per lane

// Tile grid of a row-register launch of k steps of B images (windows of win rows, wgs
// work-groups per CU): as few columns and rows of
// tiles as the window allows, then as many rows of tiles as the same number of
// rounds of work-groups takes, each shorter: a round lasts as long as one tile,
// so 3600 tiles on 512 places (8 rounds, the last of 16 tiles) cost 8 rounds
// of 48 rows and 4080 tiles cost 8 of 43 (3840x2160: 107 and 98 us).
struct RowsGeom {
    int tw, th, tiles_x, ntiles;  // ntiles: of one image
};
constexpr int kCus = 256;
inline RowsGeom hs_rows_geom(int win, int wgs, int H, int W, int k, int B) {
    RowsGeom g;
    const int mw = HS_ROWS_COLS - 2 * k, mh = win - 2 * k;
    int nx = (W + mw - 1) / mw;
    g.tw = (W + nx - 1) / nx;
    nx = (W + g.tw - 1) / g.tw;
    int ny = (H + mh - 1) / mh;
    const int64_t slots = (int64_t)wgs * kCus, col = (int64_t)nx * B;
    const int64_t rounds = (col * ny + slots - 1) / slots;
    ny = (int)std::max<int64_t>(ny, std::min<int64_t>(rounds * slots / col, H));
    g.th = (H + ny - 1) / ny;
    ny = (H + g.th - 1) / g.th;
    g.tiles_x = nx;
    g.ntiles = nx * ny;
    return g;
}

// Cost in us of a row-register launch of k steps, from what bounds it: the busiest CU
// takes m tiles, each of which loads its window (load per window row) and in each
// step pays its barrier (step) and updates its active rows (row each; tile rows
// + k - 1 on average over the steps) at 29 VALU instructions per wave-row.  Fitted
// per build to 21 image sizes from 64^2 to 3840x2160 at k = 4 .. 16, the (build, k)
// within 10 % of a size's fastest weighing most: the pair of least cost was the
// fastest measured one at 17 of them, and within 3.8 % of it at the others.
struct RowsCost {
    float launch, load, row, step;
    float us(int win, int m, int k, float active) const {
        return launch + (float)m * (load * (float)win +
                                    (float)k * (row * std::min(active, (float)win) + step));
    }
};
constexpr RowsCost kRowsCost16x2 = {2.41f, 0.0472f, 0.0103f, 0.1530f};   // waves x rows
constexpr RowsCost kRowsCost16x3 = {2.01f, 0.0468f, 0.0084f, 0.1960f};
constexpr RowsCost kRowsCost16x4 = {1.86f, 0.0484f, 0.0089f, 0.1974f};
constexpr RowsCost kRowsCost16x5 = {1.56f, 0.0488f, 0.0087f, 0.2316f};
constexpr RowsCost kRowsCost8x7 = {4.68f, 0.0152f, 0.0094f, 0.1509f};
constexpr RowsCost kRowsCost8x9 = {5.23f, 0.0166f, 0.0087f, 0.1924f};
constexpr RowsCost kRowsCost16x4two = {3.88f, 0.0235f, 0.0087f, 0.0956f};  // two per CU

// LDS of one work-group in hs_rows_tile: per wave the first and last row of its strip, double
// buffered (the neighbouring waves read them), and its other rows (read by the wave
// alone), between a wave above the first and one below the last.
template <int NW, int P>
struct HsStripLds {
    float2 wave[NW + 2][P + 2][HS_ROWS_COLS];
};
// a wave's rows in it: first and last of buffer 0, of buffer 1, the others
template <int P>
constexpr unsigned hs_strip_row(int buf, int j) {
    return 512u * (unsigned)(j == 0 ? 2 * buf : j == P - 1 ? 2 * buf + 1 : 3 + j);
}
typedef float hs_f2 __attribute__((ext_vector_type(2)));
using hs_lds_f2 = __attribute__((address_space(3))) hs_f2;
// the same for kernels that index it themselves
template <int NW, int P>
struct HsRowsLds {
    float2 edge[2][NW][2][HS_ROWS_COLS];
    float2 row[NW][P > 2 ? P - 2 : 1][HS_ROWS_COLS];
};

// Derivative planes computed by a solve's first launch itself (SETUP builds): the
// frames, the planes to write, and the weights of Dx, Dy and Dt, whose taps sit
// at the canonical offsets (hs_cube_taps).
struct HsSetup {
    const float *I1, *I2;
    float *Ix, *Iy, *It;
    float w[12];
};
// the canonical derivative stencils' offsets in their tap order: Dx and Dt, Dy
constexpr int HS_CUBE_OX[2][4] = {{0, 1, 0, 1}, {0, 0, 1, 1}};
constexpr int HS_CUBE_OY[2][4] = {{0, 0, 1, 1}, {0, 1, 0, 1}};

// 16 of a cell's 29 VALU instructions take a weight, and run at up to twice the rate
// when it is in a vector register (in_vgpr).  A build holds as many of the eight
// there as its register budget leaves; two of the two-per-CU ones, which
// have room for 2, also come as TWO builds for stencils whose first four and last
// four weights are equal (Horn and Schunck's own), which need two registers.
// Per 8 iterations, scalar weights / as many as fit / TWO: 1920x1080 (16 x 4 rows) 32.3 /
// 29.7 / 27.8 us, 2560x1440 (8 x 9) 50.4 / 47.2 / 45.2.
template <int NW, int P, bool PRE>
constexpr int kRowsVgprWeights = (NW == 16 && !PRE) || P == 9 ? 2 : 8;
template <int NW, int P, bool PRE>
constexpr bool kRowsTwoBuild = kRowsVgprWeights<NW, P, PRE> < 8;
inline bool hs_two_weights(const float *w) {
    for (int d = 1; d < 4; ++d)
        if (std::memcmp(w + d, w, 4) || std::memcmp(w + 4 + d, w + 4, 4)) return false;
    return true;
}

// a window row around one column: left neighbour, cell, right neighbour
struct HsTri {
    float2 l, c, r;
};

// Tile (txi, tyi) of the grid of tw x th tiles of image a, k steps; w: the
// averaging weights in the canonical tap order; off: the image's first element in the
// planes (of a batch).  The host keeps tw + 2k <= 64
// and th + 2k <= NW * P.
// PRE: a row's left and right neighbours for the next step are read as soon as
// the row is written, so their latency is a step away from their use (four
// more registers per row); otherwise they are read as the row is reached.
// G: rows computed together (independent fma chains in flight, one range check).
// LOUT: also store each step's (ubar, vbar) of the output tile (HsImage::lub).
// SETUP: the window's derivatives come from the frames (su), and the tile's are
// stored for the launches that follow.  A solve then needs no setup pass: that
// pass is one launch of latency for an image of any ordinary size (135x240 11
// us, 480x640 14.6 us, against 11 and 20 B/px of traffic) and this is
// 27 more VALU instructions per cell of one launch.
template <int NW, int P, bool PRE, int G, bool TWO, bool LOUT = false, bool SETUP = false>
__device__ __forceinline__ void hs_rows_tile(const HsImage &a, int txi, int tyi, int tw, int th,
                                             int k, const float (&weights)[8],
                                             HsStripLds<NW, P> &lds,
                                             const HsSetup *su = nullptr, int64_t off = 0) {
    static_assert(P >= 2, "a strip has a first and a last row");
    constexpr int WV = kRowsVgprWeights<NW, P, PRE>;
    float w[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        if (TWO)
            w[d] = d % 4 == 0 ? in_vgpr(weights[d]) : w[d / 4 * 4];
        else
            w[d] = d < WV ? in_vgpr(weights[d]) : weights[d];
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int H = a.H, W = a.W;
    const int x0 = txi * tw, y0 = tyi * th;
    const int x1 = min(x0 + tw, W), y1 = min(y0 + th, H);
    // window: columns x0 - k .., rows from y0 - k, or from the image's first
    const int gx0 = x0 - k, gy0 = max(y0 - k, 0);
    const int gx = gx0 + lane;
    const int r0 = wave * P;  // the strip's first window row
    // The strip's first image row, uniform over the wave and 64 bits, so that planes may
    // have any size; byte offsets from it fit 32 bits.  Against 32-bit offsets from the
    // image's start, 3840x2160, 500 it: 5902 -> 5804 us (the stores need no 64-bit vector
    // additions); a uniform base for every row, 10 SALU instructions a row, 5949 -> 6080.
    const int rs = min(gy0 + r0, H - 1);
    const int64_t strip = off + (int64_t)rs * W;
    const unsigned rowb = (unsigned)W * 4u;

    float cx[P], cy[P], ct[P], cd[P], cr[P], u[P], v[P];
    {
        // every load of the thread is issued before any is used
        const unsigned co = (unsigned)clampi(gx, 0, W - 1) * 4u;
        auto ld = [&](const float *plane, unsigned o) {
            return ld_g(reinterpret_cast<const float *>(
                reinterpret_cast<const char *>(plane + strip) + o));
        };
        const bool pd = a.den != nullptr;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const unsigned o = (unsigned)(min(gy0 + r0 + j, H - 1) - rs) * rowb + co;
            u[j] = ld(a.u_in, o);
            v[j] = ld(a.v_in, o);
            if (SETUP) continue;
            cx[j] = ld(a.Ix, o);
            cy[j] = ld(a.Iy, o);
            ct[j] = ld(a.It, o);
            if (pd) cd[j] = ld(a.den, o);
        }
        if constexpr (SETUP) {
            // the 2 x 2 block of each cell in both frames, its right column and
            // lower row clamped; a row is the lower row of the one above it
            const unsigned cr1 = (unsigned)min(clampi(gx, 0, W - 1) + 1, W - 1) * 4u;
            float f[P + 1][4];
#pragma unroll
            for (int j = 0; j <= P; ++j) {
                const unsigned ro = (unsigned)(min(gy0 + r0 + j, H - 1) - rs) * rowb;
                f[j][0] = ld(su->I1, ro + co);
                f[j][1] = ld(su->I1, ro + cr1);
                f[j][2] = ld(su->I2, ro + co);
                f[j][3] = ld(su->I2, ro + cr1);
            }
#pragma unroll
            for (int j = 0; j < P; ++j) {
                // stencil s (0 Dx, 1 Dy, 2 Dt) of frame q: fma in tap order from 0
                auto cube = [&](int s, int q) {
                    float acc = 0.0f;
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        acc = fmaf(su->w[4 * s + d],
                                   f[j + HS_CUBE_OY[s & 1][d]][2 * q + HS_CUBE_OX[s & 1][d]], acc);
                    return acc;
                };
                cx[j] = cube(0, 0) + cube(0, 1);
                cy[j] = cube(1, 0) + cube(1, 1);
                const float t2 = cube(2, 1), t1 = cube(2, 0);
                ct[j] = t2 - t1;
                const int gy = gy0 + r0 + j;
                if (gx >= x0 && gx < x1 && gy >= y0 && gy < y1) {
                    const unsigned o = (unsigned)j * rowb + co;  // (co: a tile's column is inside)
                    auto st = [&](float *plane, float x) {
                        *(gfloat *)(reinterpret_cast<char *>(plane + strip) + o) = x;
                    };
                    st(su->Ix, cx[j]);
                    st(su->Iy, cy[j]);
                    st(su->It, ct[j]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            if (!pd) {
                const float m1 = cx[j] * cx[j];
                const float s1 = a.alpha2 + m1;
                const float m2 = cy[j] * cy[j];
                cd[j] = s1 + m2;
            }
            cr[j] = hs_recip(cd[j]);
        }
    }
    // the lanes of the neighbouring columns, clamped to the image and the window
    const int lmin = max(-gx0, 0), lmax = min(W - 1 - gx0, HS_ROWS_COLS - 1);
    const int li = clampi(lane - 1, lmin, lmax), ri = clampi(lane + 1, lmin, lmax);
    const int jb = H - 1 - gy0 - r0;  // the image's last row, as a strip row
    const bool in = gx >= x0 && gx < x1;

    // LDS byte addresses of a row's left neighbour, cell and right neighbour in the slot of
    // the wave above: every access is one of the three plus a constant
    constexpr unsigned SLOT = 512u * (P + 2);
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)
                              reinterpret_cast<char *>(&lds) + (unsigned)wave * SLOT;
    unsigned al = base + 8u * (unsigned)li, ac = base + 8u * (unsigned)lane,
             ar = base + 8u * (unsigned)ri;
    asm volatile("" : "+v"(al), "+v"(ac), "+v"(ar));
    auto get = [](unsigned addr) {
        const hs_f2 x = *(const hs_lds_f2 *)(uintptr_t)addr;
        return make_float2(x.x, x.y);
    };
    auto put = [&](unsigned row, float x, float y) {
        const hs_f2 z = {x, y};
        *(hs_lds_f2 *)(uintptr_t)(ac + row) = z;
    };
    // the row above the window or the image is the strip's own first row, the one below
    // its last: the wave keeps a copy in the neighbouring slot (a strip that ends with
    // the image's last row has none but such rows below it)
    const bool dup_up = wave == 0, dup_down = jb == P - 1 || wave == NW - 1;
    auto put_row = [&](int buf, int j, float x, float y) {
        put(SLOT + hs_strip_row<P>(buf, j), x, y);
        if (j == 0 && dup_up) put(hs_strip_row<P>(buf, P - 1), x, y);
        if (j == P - 1 && dup_down) put(2 * SLOT + hs_strip_row<P>(buf, 0), x, y);
    };
    // a wave's LDS writes before its reads of the same row (a wavefront's LDS
    // accesses are performed in order; this keeps the compiler's order)
    auto wave_fence = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    float2 L[PRE ? P : 1], R[PRE ? P : 1];
#pragma unroll
    for (int j = 0; j < P; ++j) put_row(0, j, u[j], v[j]);
    // (a strip that never is active writes no other edge rows)
    put_row(1, 0, u[0], v[0]);
    put_row(1, P - 1, u[P - 1], v[P - 1]);
    wave_fence();
    if (PRE) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
            L[j] = get(al + SLOT + hs_strip_row<P>(0, j));
            R[j] = get(ar + SLOT + hs_strip_row<P>(0, j));
        }
    }
    // linearisation output: the lane's offset in a row, and the strip rows in the
    // output tile
    unsigned lo0 = (unsigned)gx * 4u;
    unsigned tile_rows = 0;
    if (LOUT)
        for (int j = 0; j < P; ++j)
            if (gy0 + r0 + j >= y0 && gy0 + r0 + j < y1) tile_rows |= 1u << j;
    // Steps in which the strip has active rows (the tile grown by k - it, inside the
    // image): the first `live` ones.  All its rows are updated in them; the inactive
    // ones hold values that no active row reads.  A branch per row costs copies of its old
    // and new values and its scalar tests, 5 VALU and 5 SALU instructions per row
    // with P = 4, against 1.5 rows more per strip at the window's ends.
    const int live = gy0 + r0 >= H ? 0
                                   : clampi(min(k - 1 + r0 + P - (y0 - gy0), k - 1 + y1 - gy0 - r0),
                                            0, k);
    // BOT: the image's last row is in the strip and not its last row
    auto steps = [&](auto bot_c) {
        constexpr bool BOT = decltype(bot_c)::value;
        // buf_c: the edge buffer step it reads, (it - 1) & 1; it writes the other, which
        // was last read in step it - 1, before this barrier
        auto step = [&](auto buf_c, int it) {
            constexpr int buf = decltype(buf_c)::value;
            __syncthreads();
            // (opaque per step: otherwise every row's output address is kept
            // across the loop)
            if (LOUT) asm volatile("" : "+v"(lo0));
            const int64_t lo = LOUT ? (int64_t)(it - 1) * a.lstride + strip : 0;
            auto row = [&](int j) {
                HsTri q;
                q.c = make_float2(u[j], v[j]);
                q.l = PRE ? L[PRE ? j : 0] : get(al + SLOT + hs_strip_row<P>(buf, j));
                q.r = PRE ? R[PRE ? j : 0] : get(ar + SLOT + hs_strip_row<P>(buf, j));
                return q;
            };
            // the old rows above the group (prev) and its first (cur)
            constexpr unsigned above = hs_strip_row<P>(buf, P - 1);
            constexpr unsigned below = 2 * SLOT + hs_strip_row<P>(buf, 0);
            HsTri prev = {get(al + above), get(ac + above), get(ar + above)};
            HsTri cur = row(0);
#pragma unroll
            for (int j0 = 0; j0 < P; j0 += G) {
                const int n = P - j0 < G ? P - j0 : G;
                HsTri rows[G + 1];  // old rows j0 .. j0 + n
                rows[0] = cur;
#pragma unroll
                for (int i = 1; i < n; ++i) rows[i] = row(j0 + i);
                if (j0 + n < P)
                    rows[n] = row(j0 + n < P ? j0 + n : 0);
                else
                    rows[n] = {get(al + below), get(ac + below), get(ar + below)};
                {
                    float ub[G], vb[G], s2[G], q[G];
#pragma unroll
                    for (int i = 0; i < n; ++i) {
                        const int j = j0 + i;
                        const HsTri &up = i == 0 ? prev : rows[i > 0 ? i - 1 : 0];
                        const HsTri &me = rows[i];
                        HsTri dn = rows[i + 1];
                        if (BOT && j == jb) dn = me;
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
                        ub[i] = x;
                        vb[i] = y;
                        const float m1 = cx[j] * x;
                        const float m2 = cy[j] * y;
                        const float s1 = m1 + m2;
                        s2[i] = s1 + ct[j];
                        // hs_div_fast's quotient; its range check follows
                        q[i] = hs_quotient(s2[i], cd[j], cr[j]);
                    }
                    float mx = fabsf(q[0]), mn = mx;
#pragma unroll
                    for (int i = 1; i < n; ++i) {
                        mx = __builtin_elementwise_maximum(mx, fabsf(q[i]));
                        mn = __builtin_elementwise_minimum(mn, fabsf(q[i]));
                    }
                    if (!(mn >= 0x1p-76f && mx <= 0x1p76f)) {
#pragma unroll
                        for (int i = 0; i < n; ++i) {
                            float so = s2[i];  // opaque: the divisions stay in the branch
                            asm volatile("" : "+v"(so));
                            q[i] = so / cd[j0 + i];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < n; ++i) {
                        const int j = j0 + i;
                        const float p1 = cx[j] * q[i];
                        const float p2 = cy[j] * q[i];
                        u[j] = ub[i] - p1;
                        v[j] = vb[i] - p2;
                        put_row(buf ^ 1, j, u[j], v[j]);
                    }
                    if (LOUT && in) {
#pragma unroll
                        for (int i = 0; i < n; ++i)
                            if ((tile_rows >> (j0 + i)) & 1) {
                                const unsigned o = lo0 + (unsigned)(j0 + i) * rowb;
                                *(gfloat *)(reinterpret_cast<char *>(a.lub + lo) + o) = ub[i];
                                *(gfloat *)(reinterpret_cast<char *>(a.lvb + lo) + o) = vb[i];
                            }
                    }
                    wave_fence();
                    if (PRE) {
#pragma unroll
                        for (int i = 0; i < n; ++i) {
                            L[PRE ? j0 + i : 0] = get(al + SLOT + hs_strip_row<P>(buf ^ 1, j0 + i));
                            R[PRE ? j0 + i : 0] = get(ar + SLOT + hs_strip_row<P>(buf ^ 1, j0 + i));
                        }
                    }
                }
                prev = rows[n - 1];
                cur = rows[n];
            }
        };
        // two steps a round, so that a row's old and new values change places
        // without copies and the buffers' addresses are constants
        int it = 1;
        while (it <= live) {
            step(std::integral_constant<int, 0>(), it++);
            if (it > live) break;
            step(std::integral_constant<int, 1>(), it++);
        }
        for (; it <= k; ++it) __syncthreads();
    };
    if (jb >= 0 && jb < P - 1)
        steps(std::true_type());
    else
        steps(std::false_type());
    // (plain stores: the tile's rows are partial cache lines, which the L2 merges
    // with the neighbouring tiles' before they go to memory)
    if (in) {
        unsigned so = (unsigned)gx * 4u;
        asm volatile("" : "+v"(so));  // the rows' offsets are not kept across the steps
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int gy = gy0 + r0 + j;
            if (gy >= y0 && gy < y1) {
                const unsigned o = (unsigned)j * rowb + so;
                *(gfloat *)(reinterpret_cast<char *>(a.u_out + strip) + o) = u[j];
                *(gfloat *)(reinterpret_cast<char *>(a.v_out + strip) + o) = v[j];
            }
        }
    }
}

}  // namespace hmx
