// matched_device.h - gather of the exact transpose of the Siddon forward
// projector (device code shared by the standalone transpose and the fused
// matched OSTR update).
//
// For voxel j: total = sum over the launch's views of cos(t) sum_i a_ij p_i,
// with a_ij the length of ray i (source -> bin centre, the forward
// projector's ray) inside the voxel box: the entry of the forward walk
// (Tomo_OSTR.cu:612-890) in exact arithmetic. A ray's parameter interval in a
// voxel is the intersection of three slab intervals, and within one slice and
// view they separate: the z slab is the same for all rays, the x slab depends
// on the detector column and the voxel's x only, the y slab on the detector
// row and the voxel's y only. So a wave (64 voxels along x, R rows of one
// slice) clips each candidate column once per view and lane and uses it for
// its R rows, clips each (voxel row, detector row) pair in one lane and reads
// it back with readlane, and what is left per candidate ray is a max, a min,
// the ray length and one gather. The slab reciprocals and the ray length use
// the hardware reciprocal and square root (<= 1 ulp each). The sinogram is
// detector-row-major [slot][nby][nbx], so neighbouring lanes (voxels along x)
// read neighbouring bins.
//
// Candidates are the bins whose centres lie in the voxel's shadow, widened by
// a margin that covers the rounding of the shadow (MatchedSlots::mx, my): about
// 2 rays per voxel and view for the ~1.5 that meet the voxel, where a range
// widened by a whole bin on either side had 11. Bound by VALU issue and, at
// 95 VGPRs (5 waves per SIMD), in part by the gathers' latency. With every
// candidate clipped in every lane, the fused update took 258 us at 256x256x48
// voxels and 15 views (FP16 h), now 114; one view's standalone transpose 23.4,
// now 15.6.
//
// Precision: each ray is parametrised from its detector end, p(t) = E + t (S -
// E). The volume lies next to the detector, so the clip parameters are small
// (t ~ 0.03 instead of ~0.97 from the source) and their FP32 resolution, which
// sets the error of a segment length, is ~16x finer.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "ostr_internal.h"

namespace ostr {

// Margin in bins that covers the FP32 error of a shadow end's bin coordinate
// along one axis: the end is s + (b - s) t with t = (ez - sz) / (bz - sz), each
// operand within a few 2^-24 of its magnitude, t also of the cancellation in
// bz - sz. Beyond half a bin (a source next to the volume, very fine bins) one
// bin, which covers no such error: there a ray may be left out between the exact
// and the FP32 end, and its part of the voxel is as short as the rounding of the
// slice's faces is long (3e-5 mm at 660 mm). A margin that covered it would be
// the whole detector in every slice for the sake of the uppermost, and one per
// slice and view cost 1% of the accelerated iteration.
inline float matched_margin(const DevGeom& g, const ViewTab* v, int n, bool along_x) {
    const double p0 = along_x ? g.x_p0 : g.y_p0, d0 = along_x ? g.x_d0 : g.y_d0;
    const double ext = along_x ? (double)g.nx * g.dx : (double)g.ny * g.dy;
    const double size = along_x ? g.dbx : g.dby;
    const int bins = along_x ? g.nbx : g.nby;
    const double z_lo = g.z_p0, z_hi = z_lo + (double)g.nz * g.dz;
    double worst = 0.0;
    for (int a = 0; a < n; ++a) {
        const double s = along_x ? v[a].x0 : g.src_y, sz = v[a].z0;
        const double near = std::min(sz - z_lo, sz - z_hi);
        if (!(near > 0.0)) return 1.0f;
        const double pos = std::max({std::fabs(p0), std::fabs(p0 + ext), std::fabs(s),
                                     std::fabs(d0), std::fabs(d0 + bins * size)});
        const double z = std::max({std::fabs(z_lo), std::fabs(z_hi), std::fabs(sz)});
        worst = std::max(worst, pos * (1.0 + z / near));
    }
    const double m = 0x1p-20 * (worst / size + bins);
    return m < 0.5 ? (float)m : 1.0f;
}
inline MatchedSlots matched_slots(const DevGeom& g, const ViewTab* v, int n) {
    MatchedSlots S;
    for (int a = 0; a < n; ++a) {
        S.x0[a] = v[a].x0;
        S.z0[a] = v[a].z0;
        S.c[a] = v[a].c;
    }
    S.mx = matched_margin(g, v, n, true);
    S.my = matched_margin(g, v, n, false);
    return S;
}

// Voxel rows per wave, R. More rows share a lane's clipped columns (about 35 of
// the ~80 instructions per voxel and view at R = 1), fewer keep more waves in
// flight. Fused update of 9 views, us at R = 1 / 2 / 4 by the waves at R = 1: 1920
// (120x60x16 voxels) 11.4 / 12.4 / 16.9, 8000 (200x100x20) 23.8 / 19.7 / 20.5, 12000
// (200x150x20) 31.6 / 26.8 / 25.0, 16000 (200x100x40) 39.8 / 31.4 / 29.8, 24576
// (256x256x24) 58.3 / 48.7 / 50.1, 49152 (256x256x48) 111 / 90.1 / 88.4, 792000
// (1400x600x60) 1935 / 1598 / 1587; the transpose alone at 12000 25.6 / 22.1 / 20.7,
// at 24576 45.7 / 35.6 / 31.5.
inline int matched_row_count(const DevGeom& g) {
    const int64_t waves = (int64_t)((g.nx + 63) / 64) * g.ny * g.nz;  // at R = 1
    return waves >= 10000 ? 4 : waves >= 4096 ? 2 : 1;
}
// f(std::integral_constant<int, R>) for the geometry's row count.
template <typename F>
hipError_t by_matched_rows(const DevGeom& g, F f) {
    switch (matched_row_count(g)) {
        case 4: return f(std::integral_constant<int, 4>());
        case 2: return f(std::integral_constant<int, 2>());
        default: return f(std::integral_constant<int, 1>());
    }
}

// origin + (i + 1/2) size rounded once to float: i + 1/2 is exact in FP32
// (|i| < 2^23), so the fma is the correctly rounded value. The forward walk's
// bin_centre forms the same sum in FP64 and rounds it to float; the product
// is exact in FP64 (at most 48 significant bits) and so is the sum while
// |origin| < 2^28 size (all its bits within 53 places), so the two agree, at
// a quarter of the cost (no FP64 conversions or arithmetic).
__device__ __forceinline__ float matched_bin_centre(float origin, int i, float size) {
    return fmaf((float)i + 0.5f, size, origin);
}

// The part of [z0, z1] in which the line e + t d (d = s - e) lies in [lo, hi]
// along one axis; z0 <= t0, t1 <= z1 always (finite), empty when t0 >= t1. A
// line parallel to the axis' planes (d = 0): the quotients are infinities of
// equal signs outside and of opposite signs inside, NaN on a face, which
// fminf / fmaxf drop, so a face counts as outside.
__device__ __forceinline__ void matched_slab(float e, float d, float lo, float hi, float z0,
                                             float z1, float& t0, float& t1) {
    const float inv = __builtin_amdgcn_rcpf(d);
    const float a = (lo - e) * inv, b = (hi - e) * inv;
    t0 = __builtin_amdgcn_fmed3f(fminf(a, b), z0, z1);
    t1 = __builtin_amdgcn_fmed3f(fmaxf(a, b), z0, z1);
}

// First and last candidate bin [b0, b1] along one axis for the shadow of
// [lo, hi] from source coordinate s at depth ratios ta, tb (the slice's faces).
__device__ __forceinline__ void matched_range(float lo, float hi, float s, float ta, float tb,
                                              float origin, float inv_size, float margin,
                                              int bins, int& b0, int& b1) {
    const float l = lo - s, h = hi - s;
    const float a0 = fmaf(l, ta, s), a1 = fmaf(h, ta, s);
    const float c0 = fmaf(l, tb, s), c1 = fmaf(h, tb, s);
    const float mn = fminf(fminf(a0, a1), fminf(c0, c1));
    const float mx = fmaxf(fmaxf(a0, a1), fmaxf(c0, c1));
    b0 = min(max((int)ceilf(fmaf(mn - origin, inv_size, -0.5f - margin)), 0), bins);
    b1 = min(max((int)floorf(fmaf(mx - origin, inv_size, margin - 0.5f)), -1), bins - 1);
}

__device__ __forceinline__ float matched_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// total[r] = sum over slots a of (cos_weight ? cos(t_a) : 1) sum_i a_ij P[a][i]
// for the voxels (ix, iy0 + r, iz), r < R; slot sums accumulated with fma in
// slot order. All 64 lanes of the wave call it with consecutive ix (lanes past
// nx and rows past ny get 0) and the same iy0, iz.
template <typename TP, int R>
__device__ __forceinline__ void matched_rows(const DevGeom& g, const MatchedSlots& S,
                                             int n_slots, int cos_weight,
                                             const VolReader<TP>& P, int ix, int iy0, int iz,
                                             float (&total)[R]) {
    constexpr int KI = 4;             // columns clipped at a time
    constexpr int KJ = 4;             // detector rows per voxel row held in lanes
    constexpr int VC = 64 / (R * KJ);  // views per pass over the row terms
    constexpr uint32_t E = sizeof(TP);
    const int lane = threadIdx.x & 63;
    const float bx0 = fmaf((float)ix, g.dx, g.x_p0), bx1 = fmaf((float)(ix + 1), g.dx, g.x_p0);
    const float bz0 = fmaf((float)iz, g.dz, g.z_p0), bz1 = fmaf((float)(iz + 1), g.dz, g.z_p0);
    const float sy = g.src_y, ez = -g.det_r;
    const float inv_dbx = 1.0f / g.dbx, inv_dby = 1.0f / g.dby;
    const uint32_t nbin = (uint32_t)g.nbx * g.nby;
    const bool lane_in = ix < g.nx;
    // slot a's parameters in lane a, read back with readlane
    const float lx = lane < n_slots ? S.x0[lane] : 0.0f;
    const float lz = lane < n_slots ? S.z0[lane] : 0.0f;
    const float lc = lane < n_slots ? S.c[lane] : 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) total[r] = 0.0f;

    for (int c0 = 0; c0 < n_slots; c0 += VC) {
        // Row terms: lane r + R (jj + KJ k) holds detector row jj of voxel row
        // r for slot c0 + k, its clip and its share of the squared ray length.
        const int rr = lane % R, rj = (lane / R) % KJ, ra = c0 + lane / (R * KJ);
        const float rsz = __shfl(lz, ra & 63, 64);
        const float rddz = ez - rsz;
        const float rta = rddz * __builtin_amdgcn_rcpf(bz0 - rsz);
        const float rtb = rddz * __builtin_amdgcn_rcpf(bz1 - rsz);
        float rz0, rz1;
        {
            const float inv = __builtin_amdgcn_rcpf(rsz - ez);
            const float a = (bz0 - ez) * inv, b = (bz1 - ez) * inv;
            rz0 = fminf(a, b);
            rz1 = fmaxf(a, b);
        }
        const int iy = iy0 + rr;
        const float by0 = fmaf((float)iy, g.dy, g.y_p0), by1 = fmaf((float)(iy + 1), g.dy, g.y_p0);
        int j0, j1;
        matched_range(by0, by1, sy, rta, rtb, g.y_d0, inv_dby, S.my, g.nby, j0, j1);
        const int nj = ra < n_slots && iy < g.ny ? max(j1 - j0 + 1, 0) : 0;
        const float rey = matched_bin_centre(g.y_d0, j0 + rj, g.dby);
        const float rdy = sy - rey;
        float ry0, ry1;
        matched_slab(rey, rdy, by0, by1, rz0, rz1, ry0, ry1);
        const float rdyz = fmaf(rddz, rddz, rdy * rdy);

        const int na = n_slots - c0 < VC ? n_slots - c0 : VC;
        for (int k = 0; k < na; ++k) {
            const int a = c0 + k, src = k * R * KJ;
            const float sx = matched_lane(lx, a);
            const float ta = matched_lane(rta, src), tb = matched_lane(rtb, src);
            const float tz0 = matched_lane(rz0, src), tz1 = matched_lane(rz1, src);
            int i0, i1;
            matched_range(bx0, bx1, sx, ta, tb, g.x_d0, inv_dbx, S.mx, g.nbx, i0, i1);
            if (!lane_in) i1 = i0 - 1;
            float acc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = 0.0f;
            // one group of NI columns of every lane: the rows' candidate rays
            auto rows = [&](auto ni, int ib) {
                constexpr int NI = decltype(ni)::value;
                float t0[NI], t1[NI], d[NI];
                uint32_t off[NI];
                float fi = (float)(i0 + ib) + 0.5f;
#pragma unroll
                for (int c = 0; c < NI; ++c, fi += 1.0f) {
                    const float ex = fmaf(fi, g.dbx, g.x_d0);
                    d[c] = sx - ex;
                    matched_slab(ex, d[c], bx0, bx1, tz0, tz1, t0[c], t1[c]);
                    if (i0 + ib + c > i1) t1[c] = t0[c];
                    off[c] = (uint32_t)(i0 + ib + c) * E;
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int m = __builtin_amdgcn_readlane(nj, src + r);
                    const int jb = __builtin_amdgcn_readlane(j0, src + r);
                    for (int jj = 0; jj < m; ++jj) {
                        float y0, y1, dyz;
                        if (jj < KJ) {
                            const int l = src + r + R * jj;
                            y0 = matched_lane(ry0, l);
                            y1 = matched_lane(ry1, l);
                            dyz = matched_lane(rdyz, l);
                        } else {  // more rows in the shadow than lanes hold
                            const float ey = matched_bin_centre(g.y_d0, jb + jj, g.dby);
                            const float dy = sy - ey, sz = matched_lane(lz, a);
                            matched_slab(ey, dy, fmaf((float)(iy0 + r), g.dy, g.y_p0),
                                         fmaf((float)(iy0 + r + 1), g.dy, g.y_p0), tz0, tz1, y0,
                                         y1);
                            dyz = fmaf(ez - sz, ez - sz, dy * dy);
                        }
                        // wave-uniform: rides in the load's scalar offset
                        const uint32_t row =
                            ((uint32_t)a * nbin + (uint32_t)(jb + jj) * (uint32_t)g.nbx) * E;
                        float w[NI], p[NI];
#pragma unroll
                        for (int c = 0; c < NI; ++c) {
                            const float u0 = fmaxf(t0[c], y0), u1 = fminf(t1[c], y1);
                            w[c] = u1 - u0;
                            // an empty candidate reads past the buffer's end: 0
                            p[c] = P.at_byte(u0 < u1 ? off[c] : 0xFFFFFFF0u, row);
                        }
#pragma unroll
                        for (int c = 0; c < NI; ++c) {
                            const float len = __builtin_amdgcn_sqrtf(fmaf(d[c], d[c], dyz));
                            acc[r] = fmaf(w[c] * len, p[c], acc[r]);
                        }
                    }
                }
            };
            for (int ib = 0; __any(i0 + ib <= i1); ib += KI) {
                if (!__any(i0 + ib + 1 <= i1))
                    rows(std::integral_constant<int, 1>(), ib);
                else if (!__any(i0 + ib + 2 <= i1))
                    rows(std::integral_constant<int, 2>(), ib);
                else if (!__any(i0 + ib + 3 <= i1))
                    rows(std::integral_constant<int, 3>(), ib);
                else
                    rows(std::integral_constant<int, 4>(), ib);
            }
            const float cw = cos_weight ? matched_lane(lc, a) : 1.0f;
#pragma unroll
            for (int r = 0; r < R; ++r) total[r] = fmaf(cw, acc[r], total[r]);
        }
    }
}

}  // namespace ostr
