// sbp_device.h - device code of the voxel-driven bilinear backprojector (SBP),
// the sliding-window prior and the OSTR update, shared by the standalone
// backprojector, the OS-SART updates, the fused and the batched OSTR updates.
//
// SBP follows backprj_gpu_manyviews_SBP (Tomo_OSTR.cu:1553-1734): the voxel
// centre is projected from the source onto the detector plane z = -detectorR;
// the bilinear taps (ilb,jlb) are chosen with the reference's half-bin rule and
// masked one by one to the detector; the interpolated value is scaled by
// Vsize_z * |S|^2/|S-V|^2 and summed over the slots of the launch, in slot
// order. The ray parameter t and the tap positions use the reference's exact
// divisions (a 1-ulp change of a tap position at bin ~200 is 1.5e-5 of a bin,
// visible on rough data); only the depth-weight division is a hardware
// reciprocal (a factor within ~1 ulp).
//
// MI355X mapping. The kernels read the sinogram in detector-row-major layout
// [slot][nby][nbx] (x fastest) and put the 64 lanes of a wave on 64
// consecutive voxels along x, so a wave's taps fall on ~50 consecutive bins of
// one or two detector rows (a few cache lines). Because every voxel of one
// slice sees the same ray parameter t, the tap column (ilb, fracI) depends
// only on (x, slice, view) and the tap row (jlb, fracJ) only on (y, slice,
// view): a lane computes its column terms once per view and reuses them for
// the ROWS rows it owns, and the row terms are wave-uniform. Work-group tiles
// (64 x ROWS NW voxels of one slice, NW waves) are dealt to XCDs in contiguous
// ranges.
//
// The fused update computes, per voxel and in one pass,
//   capL = M * SBP(h)                      (Tomo_OSTR_gold.cpp:759-771)
//   RD, RDD = prior(x_in)                  (:775)
//   x_out = max(0, x - (capL + b RD)/(d + 2 b RDD))   (update_est :265-295)
// reading x_in and writing x_out (double-buffered, so the prior sees the
// pre-update image as the reference's sequential order does).
#pragma once

#include <type_traits>

#include "prior_device.h"

namespace ostr {

// Tile shape: R voxel rows (y) per wave, NW waves per work-group, 64 voxels
// along x, one slice. The single-case kernels have CASE_WAVES waves and the
// rows of by_sbp_rows, the batched kernels take the shape from their caller.
// The waves of a group share nothing, and a group's registers are free for the
// next one only when its last wave ends: with 4, 2 and 1 waves a clinical
// iteration took 2850 / 2817 / 2794 us, the accelerated one at 200x100x20 38.6 /
// 37.2 / 37.4, at 256x256x48 173.1 / 174.9 / 172.3.
constexpr int CASE_WAVES = 1;
constexpr int TILE_X = 64;
// prior_rows modes (by_prior_mode)
constexpr int PRIOR_INTERIOR = 0, PRIOR_EDGE = 1, PRIOR_GENERIC = 2;

__device__ __forceinline__ float cell_centre(float origin, int i, float size) {
    return (float)((double)origin + ((double)i + 0.5) * (double)size);
}

// Half-bin tap rule of Tomo_OSTR.cu:1668-1678.
__device__ __forceinline__ void tap(float m, int& l, float& f) {
    l = (int)floorf(m);
    if (m < (float)l + 0.5f) l -= 1;
    f = m - ((float)l + 0.5f);
}

struct TileCoord {
    int ix, iy0, iz;
};

// Voxel coordinates of this thread in volume tile t (x tiles fastest, then y
// tiles, then slices); the wave owns rows iy0 .. iy0+R-1.
template <int R, int NW>
__device__ __forceinline__ TileCoord tile_coord(const DevGeom& g, int t) {
    constexpr int TILE_Y = R * NW;
    const int tiles_x = (g.nx + TILE_X - 1) / TILE_X;
    const int tiles_y = (g.ny + TILE_Y - 1) / TILE_Y;
    const int bx = t % tiles_x;
    const int rest = t / tiles_x;
    TileCoord c;
    c.ix = bx * TILE_X + (threadIdx.x & 63);
    c.iy0 = (rest % tiles_y) * TILE_Y + (threadIdx.x >> 6) * R;
    c.iz = rest / tiles_y;
    return c;
}

__device__ __forceinline__ float readlane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// total[r] = sum over slots of the SBP value of voxel (ix, iy0 + r, iz);
// prj is [slot][nby][nbx], read through a buffer resource with 32-bit element
// offsets. The row terms (jlb, fracJ, y offset) of a (row, slot) pair are
// wave-uniform: lane r + ROWS*k evaluates them for row r and slot k of a chunk
// of VIEW_CHUNK slots, and every lane reads them back with readlane, so each
// exact division runs once per wave. When every lane's two tap columns and the
// row's two tap rows lie on the detector (the common case), the four taps are
// loaded without masks; otherwise each tap is masked on its own, as the
// reference does.
// SENS: also sens[r] = sum over slots of the same bilinear weights applied to
// the valid taps' indicator (the OS-SART sensitivity, backprj_OSSART_gpu_
// manyviews, Tomo_OSTR.cu:1856-1888), scaled like the data term.
template <typename TP, int ROWS, bool SENS = false>
__device__ __forceinline__ void sbp_rows(const DevGeom& g, const SlotTab& S, int n,
                                         const VolReader<TP>& P, int ix, int iy0, int iz,
                                         float total[ROWS], float* sens = nullptr) {
    constexpr int VIEW_CHUNK = 64 / ROWS;
    const uint32_t nbin = (uint32_t)g.nbx * (uint32_t)g.nby;
    const uint32_t nbx = (uint32_t)g.nbx;
    const int lane = threadIdx.x & 63;
    const float y0 = g.src_y;
    const float x1 = cell_centre(g.x_p0, ix, g.dx);
    const float z1 = cell_centre(g.z_p0, iz, g.dz);
    // slot parameters: lane a holds slot a (n <= 64); the loops below take
    // them with readlane (uniform) or shfl (per lane), no memory reads
    const float sx0 = lane < n ? S.x0[lane] : 0.0f;
    const float sz0 = lane < n ? S.z0[lane] : 0.0f;
    const float snum = lane < n ? S.num[lane] : 0.0f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        total[r] = 0.0f;
        if (SENS) sens[r] = 0.0f;
    }
    for (int c0 = 0; c0 < n; c0 += VIEW_CHUNK) {
        int rt_jl = -2;
        float rt_fj = 0.0f, rt_ey = 0.0f, rt_t = 0.0f;
        {
            const int r = lane % ROWS, a = c0 + lane / ROWS;
            const float z0 = __shfl(sz0, a & 63, 64);
            if (a < n) {
                const float y1 = cell_centre(g.y_p0, iy0 + r, g.dy);
                rt_ey = y0 - y1;
                if (z1 != z0) {
                    const float t = (-g.det_r - z0) / (z1 - z0);
                    rt_t = t;
                    const float y2 = fmaf(y1 - y0, t, y0);
                    tap((y2 - g.y_d0) / g.dby, rt_jl, rt_fj);
                }
            }
        }
        const int na = n - c0 < VIEW_CHUNK ? n - c0 : VIEW_CHUNK;
        // y0 - y1 of row r does not depend on the view: read once per chunk
        float eyr[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) eyr[r] = readlane_f(rt_ey, r);
        for (int k = 0; k < na; ++k) {
            const int a = c0 + k;
            const float x0 = readlane_f(sx0, a), z0 = readlane_f(sz0, a);
            const float num = readlane_f(snum, a);
            if (z1 == z0) continue;
            const float ex = x0 - x1, ez = z0 - z1;
            const float exx = ex * ex;
            // the view's ray parameter (the slice's, the same for every lane):
            // row 0's row-term lane divided it already
            const float t = readlane_f(rt_t, k * ROWS);
            const float x2 = fmaf(x1 - x0, t, x0);
            int il;
            float fi;
            tap((x2 - g.x_d0) / g.dbx, il, fi);
            const bool i0 = (unsigned)il < (unsigned)g.nbx;
            const bool i1 = (unsigned)(il + 1) < (unsigned)g.nbx;
            const bool wave_i_ok = __all(i0 && i1);
            const float omfi = 1.0f - fi;
            const uint32_t base = (uint32_t)a * nbin + (uint32_t)il;
            // Common case: every lane's two columns and every row's two rows
            // on the detector. Then the taps of all ROWS rows are loaded in
            // one straight run (2 ROWS loads in flight) before any is used;
            // with a per-row choice of load form each row's loads would wait
            // for the previous row's. Same operations in the same order as
            // the per-row form below, so the same bits.
            bool all_rows = wave_i_ok;
            int jlr[ROWS];  // wave-uniform
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const int jl = __builtin_amdgcn_readlane(rt_jl, k * ROWS + r);
                all_rows = all_rows && (unsigned)jl < (unsigned)g.nby &&
                           (unsigned)(jl + 1) < (unsigned)g.nby &&
                           (sizeof(TP) == 4 || a + 1 < n || jl + 2 < g.nby);
                jlr[r] = jl;
            }
            if (all_rows) {
                float p[ROWS][4];
                if constexpr (sizeof(TP) == 4) {
                    // the row's offset jl nbx is wave-uniform: it rides in the
                    // scalar offset, the lane's column in the vector offset
                    const uint32_t vb = base * 4u;
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) {
                        const uint32_t jl = (uint32_t)jlr[r];
                        P.pair_bytes(vb, jl * nbx * 4u, p[r][0], p[r][1]);
                        P.pair_bytes(vb, (jl + 1u) * nbx * 4u, p[r][2], p[r][3]);
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) {
                        const uint32_t off = base + (uint32_t)jlr[r] * nbx;
                        P.pair(off, p[r][0], p[r][1]);
                        P.pair(off + nbx, p[r][2], p[r][3]);
                    }
                }
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    const int src = k * ROWS + r;
                    const float fj = readlane_f(rt_fj, src);
                    const float ey = eyr[r];
                    const float den = fmaf(ez, ez, fmaf(ey, ey, exx));
                    const float dw = num * __builtin_amdgcn_rcpf(den);
                    float d1 = omfi * p[r][0];
                    d1 = fmaf(fi, p[r][1], d1);
                    float d2 = omfi * p[r][2];
                    d2 = fmaf(fi, p[r][3], d2);
                    float u = fmaf(fj, d2, (1.0f - fj) * d1);
                    u = (u * g.dz) * dw;
                    total[r] = total[r] + u;
                    if (SENS) {
                        // every tap valid: d1_sen = d2_sen = (1-fI) + fI
                        const float d1s = omfi + fi;
                        float us = fmaf(fj, d1s, (1.0f - fj) * d1s);
                        us = (us * g.dz) * dw;
                        sens[r] = sens[r] + us;
                    }
                }
                continue;
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const int src = k * ROWS + r;
                const int jl = __builtin_amdgcn_readlane(rt_jl, src);
                const float fj = readlane_f(rt_fj, src);
                const float ey = readlane_f(rt_ey, src);
                const bool j0 = (unsigned)jl < (unsigned)g.nby;
                const bool j1 = (unsigned)(jl + 1) < (unsigned)g.nby;
                const float den = fmaf(ez, ez, fmaf(ey, ey, exx));
                const float dw = num * __builtin_amdgcn_rcpf(den);
                const uint32_t off = base + (uint32_t)jl * nbx;
                float p00, p10, p01, p11;
                // both columns and rows on the detector: the two taps of a
                // row as one pair (one load for 16-bit h; the pair of row
                // jl + 1 may read one element past its end, which exists
                // unless that row is the last of the last slot)
                if (wave_i_ok && j0 && j1 &&
                    (sizeof(TP) == 4 || a + 1 < n || jl + 2 < g.nby)) {
                    P.pair(off, p00, p10);
                    P.pair(off + nbx, p01, p11);
                } else if (wave_i_ok && j0 && j1) {
                    p00 = P(off);
                    p10 = P(off + 1);
                    p01 = P(off + nbx);
                    p11 = P(off + nbx + 1);
                } else {
                    p00 = (i0 && j0) ? P(off) : 0.0f;
                    p10 = (i1 && j0) ? P(off + 1) : 0.0f;
                    p01 = (i0 && j1) ? P(off + nbx) : 0.0f;
                    p11 = (i1 && j1) ? P(off + nbx + 1) : 0.0f;
                }
                float d1 = omfi * p00;
                d1 = fmaf(fi, p10, d1);
                float d2 = omfi * p01;
                d2 = fmaf(fi, p11, d2);
                float u = fmaf(fj, d2, (1.0f - fj) * d1);
                u = (u * g.dz) * dw;
                total[r] = total[r] + u;
                if (SENS) {
                    // d1_sen = (1-fI)[tap 00] + fI[tap 10], likewise d2_sen
                    const float d1s = ((i0 && j0) ? omfi : 0.0f) + ((i1 && j0) ? fi : 0.0f);
                    const float d2s = ((i0 && j1) ? omfi : 0.0f) + ((i1 && j1) ? fi : 0.0f);
                    float us = fmaf(fj, d2s, (1.0f - fj) * d1s);
                    us = (us * g.dz) * dw;
                    sens[r] = sens[r] + us;
                }
            }
        }
    }
}

// Prior terms of the ROWS voxels (ix, iy0 + r, iz), r = 0..ROWS-1, from a
// sliding 3x3x3 window: each step loads the 9 values (3 slices x 3 columns) of
// the next row, so a thread reads 9*(ROWS+2) values instead of 26*ROWS. The
// 26 neighbours are visited in the reference's order (dz outer, dy, dx inner)
// and summed per weight class: a[c] = sum r(t), b[c] = sum r(t) t (prior_r:
// omega = |delta| r with |delta| in the class weights), then
// rdd = sum_c w_c a[c], rd = init(r) + sum_c w_c b[c], the same terms
// w_k omega(t) and w_k omega(t) t as the reference's per-neighbour sums with
// one weight multiply per class instead of one per neighbour and no t/delta;
// then epi(r, vi, x_centre, rdd, rd) is called for each voxel inside the
// volume. MODE (prior_mode): PRIOR_INTERIOR, the window stays inside the
// volume; otherwise a neighbour outside the volume contributes t = 0 (it is
// replaced by the voxel itself, Tomo_OSTR.cu:238-241), and PRIOR_GENERIC also
// takes k < 0.
template <int POT, int MODE, typename TI, int ROWS, typename Init, typename Epi>
__device__ __forceinline__ void prior_rows(const DevGeom& g, const VolReader<TI>& X,
                                           const TileCoord& c, const PriorClass& W,
                                           float inv_delta, Init init, Epi epi) {
    constexpr bool CHECKED = MODE != PRIOR_INTERIOR;
    const int ix = c.ix, iy0 = c.iy0, iz = c.iz;
    const uint32_t nx = g.nx, plane = (uint32_t)g.nx * g.ny;
    bool cx[3], cz[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        cx[q] = (unsigned)(ix + q - 1) < (unsigned)g.nx;
        cz[q] = (unsigned)(iz + q - 1) < (unsigned)g.nz;
    }
    float win[3][3][3];  // [row dy][slice dz][column dx]
    bool ok[3][3][3];
    auto load_row = [&](int slot, int y) {
        const bool cy = (unsigned)y < (unsigned)g.ny;
#pragma unroll
        for (int dz = 0; dz < 3; ++dz) {
            const uint32_t o = (uint32_t)(iz + dz - 1) * plane + (uint32_t)y * nx + (uint32_t)ix;
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                if (CHECKED) {
                    ok[slot][dz][dx] = cy && cz[dz] && cx[dx];
                    win[slot][dz][dx] = ok[slot][dz][dx] ? X(o + dx - 1) : 0.0f;
                } else {
                    win[slot][dz][dx] = X(o + dx - 1);
                }
            }
        }
    };
    load_row(0, iy0 - 1);
    load_row(1, iy0);
    const bool lane_ok = ix < g.nx;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        load_row(2, iy0 + r + 1);
        const float xc = win[1][1][1];
        const int iy = iy0 + r;
        const bool store = lane_ok && iy < g.ny;
        float a[5], b[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) a[k] = b[k] = 0.0f;
#pragma unroll
        for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const int nidx = dz * 9 + dy * 3 + dx;
                    if (nidx == 13) continue;
                    float t = xc - win[dy][dz][dx];
                    if (CHECKED) t = ok[dy][dz][dx] ? t : 0.0f;
                    const float rt = prior_r<POT, MODE != PRIOR_GENERIC>(t, W.k, inv_delta);
                    const int k = prior_class(nidx);
                    a[k] = a[k] + rt;
                    b[k] = fmaf(rt, t, b[k]);
                }
        float rdd = 0.0f, rd = init(r, store);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            rdd = fmaf(W.w[k], a[k], rdd);
            rd = fmaf(W.w[k], b[k], rd);
        }
        if (store) epi(r, (uint32_t)iz * plane + (uint32_t)iy * nx + (uint32_t)ix, xc, rdd, rd);
#pragma unroll
        for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                win[0][dz][dx] = win[1][dz][dx];
                win[1][dz][dx] = win[2][dz][dx];
                if (CHECKED) {
                    ok[0][dz][dx] = ok[1][dz][dx];
                    ok[1][dz][dx] = ok[2][dz][dx];
                }
            }
    }
}

// Calls f(std::integral_constant<int, MODE>) with the prior_rows mode of the
// wave (wave-uniform): PRIOR_INTERIOR when the 3x3x3 neighbourhoods of its R
// rows stay inside the volume and k >= 0, PRIOR_EDGE when only k >= 0,
// PRIOR_GENERIC otherwise.
template <int R, typename F>
__device__ __forceinline__ void by_prior_mode(const DevGeom& g, const TileCoord& c,
                                              const PriorClass& W, F f) {
    const int x_first = c.ix - (threadIdx.x & 63);
    const bool inside = x_first >= 1 && x_first + 64 < g.nx && c.iy0 >= 1 &&
                        c.iy0 + R < g.ny && c.iz >= 1 && c.iz + 1 < g.nz;
    if (W.k < 0.0f)
        f(std::integral_constant<int, PRIOR_GENERIC>());
    else if (inside)
        f(std::integral_constant<int, PRIOR_INTERIOR>());
    else
        f(std::integral_constant<int, PRIOR_EDGE>());
}

// Prior terms and SQS update of the ROWS voxels (the OSTR epilogue of the
// fused update): capL = M (0 + total), x = max(0, x - (capL + beta rd) /
// (d + 2 beta rdd)); guard: keep x where the denominator is 0.
template <int POT, int MODE, typename TI, int ROWS>
__device__ __forceinline__ void update_rows(const DevGeom& g, const VolReader<TI>& X,
                                            const VolWriter<TI>& XO, const VolReader<float>& D,
                                            const TileCoord& c, const float total[ROWS],
                                            const PriorClass& W, float inv_delta, float beta,
                                            float capl_scale, int guard) {
    const float two_beta = 2.0f * beta;
    prior_rows<POT, MODE, TI, ROWS>(
        g, X, c, W, inv_delta, [](int, bool) { return 0.0f; },
        [&](int r, uint32_t vi, float xc, float rdd, float rd) {
            // capL: 0 + total, then * M (float), as the reference host does
            const float capl = capl_scale * (0.0f + total[r]);
            const float num = capl + beta * rd;
            const float den = D(vi) + two_beta * rdd;
            float xn;
            if (guard && den == 0.0f) {
                xn = xc;
            } else {
                xn = xc - num / den;
                xn = xn < 0.0f ? 0.0f : xn;
            }
            XO(vi, xn);
        });
}

// Fused update of volume tile t (R rows per wave, NW waves per work-group).
template <int POT, typename TI, typename TP, int R, int NW>
__device__ __forceinline__ void update_tile(const DevGeom& g, const SlotTab& S, int n_slots,
                                            const TP* __restrict__ hsub,
                                            const TI* __restrict__ x_in, TI* __restrict__ x_out,
                                            const float* __restrict__ d, const PriorClass& W,
                                            float inv_delta, float beta, float capl_scale,
                                            int guard, int t) {
    const TileCoord c = tile_coord<R, NW>(g, t);
    if (c.iy0 >= g.ny) return;  // see sbp_kernel
    const uint32_t nvox = (uint32_t)g.nx * g.ny * g.nz;
    const VolReader<TP> P(hsub, (uint32_t)n_slots * g.nbx * g.nby);
    const VolReader<TI> X(x_in, nvox);
    const VolWriter<TI> XO(x_out, nvox);
    const VolReader<float> D(d, nvox);
    float total[R];
    sbp_rows<TP, R>(g, S, n_slots, P, c.ix, c.iy0, c.iz, total);
    by_prior_mode<R>(g, c, W, [&](auto m) {
        update_rows<POT, decltype(m)::value, TI, R>(g, X, XO, D, c, total, W, inv_delta, beta,
                                                    capl_scale, guard);
    });
}

inline unsigned volume_tiles(const DevGeom& g, int tile_y) {
    const int64_t tx = (g.nx + TILE_X - 1) / TILE_X, ty = (g.ny + tile_y - 1) / tile_y;
    return (unsigned)(tx * ty * g.nz);
}

// f(std::integral_constant<int, R>) with R voxel rows per wave for the
// geometry, R <= MOST. More rows share a lane's tap columns and the prior's
// window (about 20 + 9 of the ~330 issue slots per voxel at R = 8), fewer keep
// more waves in flight. By the waves the volume makes at R = 1: 2 rows below
// 16000, 8 from `line` on. update_fused of 3 views, FP32, hyperbola, us at R = 2 /
// 4 / 8: 1920 waves (120x60x16 voxels) 9.8 / 9.2 / 12.2, 8000 (200x100x20) 11.7 /
// 12.2 / 17.4, 12000 (200x150x20) 15.5 / 13.9 / 19.4, 24576 (256x256x24) 21.4 /
// 20.6 / 23.4, 49152 (256x256x48) 39.0 / 36.3 / 41.0, 99000 (600x300x33) 66.9 /
// 58.7 / 58.8, 150183 (701x333x41) 97.8 / 82.7 / 81.9, 208000 (800x400x40) 133 /
// 114 / 112, 360000 (1000x500x45) 235 / 194 / 186. Around 16000 more views favour
// fewer rows: 25 views and q2 at 12000 40.2 / 44.1 / 65.9 (the backprojection alone
// 35.7 / 39.6 / 58.6), at 16000 51.0 / 51.1 / 73.3.
constexpr int SBP_ROWS_LINE = 200000;
template <int MOST, typename F>
hipError_t by_sbp_rows(const DevGeom& g, int64_t line, F f) {
    const int64_t waves = (int64_t)((g.nx + TILE_X - 1) / TILE_X) * g.ny * g.nz;
    if (waves < 16000) return f(std::integral_constant<int, 2>());
    if (MOST < 8 || waves < line) return f(std::integral_constant<int, 4>());
    return f(std::integral_constant<int, MOST>());
}

}  // namespace ostr
