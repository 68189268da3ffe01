// backproject.hip - the voxel-driven bilinear backprojector (SBP), the OS-SART
// updates, the batched OSTR update and the dispatch of the fused ones
// (update_kernels.h) for gfx950. The device code is in sbp_device.h.
//
// The fused update computes, per voxel and in one pass,
//   capL = M * SBP(h)                      (Tomo_OSTR_gold.cpp:759-771)
//   RD, RDD = prior(x_in)                  (:775)
//   x_out = max(0, x - (capL + b RD)/(d + 2 b RDD))   (update_est :265-295)
// reading x_in and writing x_out (double-buffered, so the prior sees the
// pre-update image as the reference's sequential order does).
#include "matched_device.h"
#include "sbp_device.h"

namespace ostr {

namespace {

template <typename TP, int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void sbp_kernel(DevGeom g, SlotTab S, int n_slots,
                                                  const TP* __restrict__ prj,
                                                  float* __restrict__ img) {
    const TileCoord c = tile_coord<R, CASE_WAVES>(g, xcd_tile(blockIdx.x, gridDim.x));
    // whole waves past the last row leave; lanes past the last column stay
    // (they evaluate row terms other lanes read) and only skip the stores
    if (c.iy0 >= g.ny) return;
    const VolReader<TP> P(prj, (uint32_t)n_slots * g.nbx * g.nby);
    float total[R];
    sbp_rows<TP, R>(g, S, n_slots, P, c.ix, c.iy0, c.iz, total);
    if (c.ix >= g.nx) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int iy = c.iy0 + r;
        if (iy >= g.ny) break;
        const int64_t vi = ((int64_t)c.iz * g.ny + iy) * g.nx + c.ix;
        img[vi] = img[vi] + total[r];
    }
}

// OS-SART backprojection and update (backprj_OSSART_gpu_manyviews and the _R
// variant with a prior, Tomo_OSTR.cu:1737-2143): per voxel, u = sum / sens
// over the launch's slots (0 where sens == 0), then, in place,
//   x = max(0, x + lambda * u)                          (PRIOR false)
//   x = max(0, x + lambda * (u + beta * prior / sens))  (PRIOR true; the sign is
//                                                        the reference's)
template <typename TP, bool PRIOR, int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void sart_update_kernel(DevGeom g, SlotTab S, int n_slots,
                                                          const TP* __restrict__ diff,
                                                          float* __restrict__ img,
                                                          const float* __restrict__ prior,
                                                          float lambda, float beta) {
    const TileCoord c = tile_coord<R, CASE_WAVES>(g, group_tile());
    if (c.iy0 >= g.ny || c.iz >= g.nz) return;  // see sbp_kernel
    const VolReader<TP> P(diff, (uint32_t)n_slots * g.nbx * g.nby);
    float total[R], sens[R];
    sbp_rows<TP, R, true>(g, S, n_slots, P, c.ix, c.iy0, c.iz, total, sens);
    if (c.ix >= g.nx) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int iy = c.iy0 + r;
        if (iy >= g.ny) break;
        const int64_t vi = ((int64_t)c.iz * g.ny + iy) * g.nx + c.ix;
        float u = 0.0f, bt = 0.0f;
        if (sens[r] != 0.0f) {
            u = total[r] / sens[r];
            if (PRIOR) bt = (beta * prior[vi]) / sens[r];
        }
        const float xn = fmaf(lambda, PRIOR ? u + bt : u, img[vi]);
        img[vi] = xn < 0.0f ? 0.0f : xn;
    }
}

// The SART prior G_Huber_prior (Tomo_OSTR.cu:258-325), accumulating:
//   prior[v] += sum over the 26 neighbours of w d / sqrt(1 + (d/delta)^2),
// d = x[v] - x[neighbour] (0 for neighbours outside the volume), w = 1/distance
// in voxel-index units (no z-size ratio). This is the hyperbola gradient term
// rd of the OSTR prior with rho = 1, evaluated in FP32 (rsq of 1 + q^2, the
// terms added in the reference's order from prior[v]); the reference forms
// each term in double and rounds the sum to float after every term.
template <int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void huber_prior_kernel(DevGeom g, PriorClass W,
                                                          float inv_delta,
                                                          const float* __restrict__ x,
                                                          float* __restrict__ prior) {
    const TileCoord c = tile_coord<R, CASE_WAVES>(g, xcd_tile(blockIdx.x, gridDim.x));
    if (c.iy0 >= g.ny) return;  // see sbp_kernel
    const uint32_t nvox = (uint32_t)g.nx * g.ny * g.nz;
    const VolReader<float> X(x, nvox);
    const VolReader<float> PR(prior, nvox);
    const VolWriter<float> PW(prior, nvox);
    const uint32_t row0 = ((uint32_t)c.iz * g.ny + (uint32_t)c.iy0) * g.nx + (uint32_t)c.ix;
    auto init = [&](int r, bool store) { return store ? PR(row0 + (uint32_t)r * g.nx) : 0.0f; };
    auto epi = [&](int, uint32_t vi, float, float, float rd) { PW(vi, rd); };
    by_prior_mode<R>(g, c, W, [&](auto m) {
        prior_rows<OSTR_PRIOR_HYPERBOLA, decltype(m)::value, float, R>(g, X, c, W,
                                                                              inv_delta, init, epi);
    });
}

// Fused OS-SART subset update (the backprj_OSSART[_R] update with the Huber
// prior evaluated in the same pass): per voxel, total and sens as
// sart_update_kernel, prior = 0 + the Huber terms of x_in, then
// x_out = max(0, x_in + lambda (total/sens [+ beta prior/sens])). Reading
// x_in and writing x_out keeps the prior's neighbours at their pre-update
// values, as the separate prior launch does.
template <bool PRIOR, int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void sart_update_fused_kernel(
    DevGeom g, SlotTab S, int n_slots, const float* __restrict__ diff,
    const float* __restrict__ x_in, float* __restrict__ x_out, PriorClass W, float inv_delta,
    float lambda, float beta) {
    const TileCoord c = tile_coord<R, CASE_WAVES>(g, group_tile());
    if (c.iy0 >= g.ny || c.iz >= g.nz) return;  // see sbp_kernel
    const uint32_t nvox = (uint32_t)g.nx * g.ny * g.nz;
    const VolReader<float> P(diff, (uint32_t)n_slots * g.nbx * g.nby);
    const VolReader<float> X(x_in, nvox);
    const VolWriter<float> XO(x_out, nvox);
    float total[R], sens[R];
    sbp_rows<float, R, true>(g, S, n_slots, P, c.ix, c.iy0, c.iz, total, sens);
    auto epi = [&](int r, uint32_t vi, float xc, float, float rd) {
        float u = 0.0f, bt = 0.0f;
        if (sens[r] != 0.0f) {
            u = total[r] / sens[r];
            if (PRIOR) bt = (beta * rd) / sens[r];
        }
        const float xn = fmaf(lambda, PRIOR ? u + bt : u, xc);
        XO(vi, xn < 0.0f ? 0.0f : xn);
    };
    if (PRIOR) {
        auto init = [](int, bool) { return 0.0f; };
        by_prior_mode<R>(g, c, W, [&](auto m) {
            prior_rows<OSTR_PRIOR_HYPERBOLA, decltype(m)::value, float, R>(
                g, X, c, W, inv_delta, init, epi);
        });
    } else {
        if (c.ix >= g.nx) return;
        const uint32_t plane = (uint32_t)g.nx * g.ny;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int iy = c.iy0 + r;
            if (iy >= g.ny) break;
            const uint32_t vi = (uint32_t)c.iz * plane + (uint32_t)iy * g.nx + (uint32_t)c.ix;
            epi(r, vi, X(vi), 0.0f, 0.0f);
        }
    }
}

// Batched fused update: every case of the table in one launch. LOOP: a
// persistent grid (a fixed number of groups per CU, each looping over its
// share of the tiles, see BatchWalk); otherwise the grid gives every XCD at
// least as many groups as it has tiles and each group takes at most one, so
// the walk's state is not live across the tile (scalar registers the tile
// would otherwise spill). The case's scalars are read from the read-only case
// table with uniform addresses (scalar loads).
template <int POT, typename TI, typename TP, int R, int NW, bool LOOP>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(5))) void batch_update_kernel(
    const BatchCase* __restrict__ cases, const int* __restrict__ sched, int n_cases) {
    BatchWalk walk(sched, n_cases);
    int t, c;
    while (walk.next(t, c)) {
        const BatchCase& bc = cases[c];
        update_tile<POT, TI, TP, R, NW>(
            bc.g, bc.S, bc.n_slots, (const TP*)bc.h, (const TI*)bc.x_in, (TI*)bc.x_out, bc.d,
            bc.W, bc.inv_delta, bc.beta, bc.capl_scale, bc.guard, t);
        if (!LOOP) break;
    }
}

// [slot][nbx][nby] -> [slot][nby][nbx], TxT tiles through LDS. A thread's loads
// are all issued before the first is stored (waiting for each in turn, 9 views
// of 2048x1664 FP32 bins took 41.5 us, now 35.7; 3 views 18.6, now 12.8).
template <typename T, int TILE>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ src,
                                                        T* __restrict__ dst, int nbx, int nby) {
    constexpr int STEP = 256 / TILE, N = TILE / STEP;
    __shared__ T tile[TILE][TILE + 1];
    const int slot = blockIdx.z;
    const int i0 = blockIdx.y * TILE, j0 = blockIdx.x * TILE;
    const T* s = src + (int64_t)slot * nbx * nby;
    T* o = dst + (int64_t)slot * nbx * nby;
    const int lane = threadIdx.x % TILE, w = threadIdx.x / TILE;
    T v[N];
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int i = min(i0 + w + STEP * q, nbx - 1), j = min(j0 + lane, nby - 1);
        v[q] = s[(int64_t)i * nby + j];
    }
#pragma unroll
    for (int q = 0; q < N; ++q) tile[w + STEP * q][lane] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int j = j0 + w + STEP * q, i = i0 + lane;
        if (i < nbx && j < nby) o[(int64_t)j * nbx + i] = tile[lane][w + STEP * q];
    }
}

template <typename T, int TILE>
hipError_t transpose_t(const void* src, void* dst, int n_slots, int nbx, int nby,
                       hipStream_t st) {
    const dim3 grid((nby + TILE - 1) / TILE, (nbx + TILE - 1) / TILE, n_slots);
    hipLaunchKernelGGL((transpose_kernel<T, TILE>), grid, dim3(256), 0, st, (const T*)src, (T*)dst,
                       nbx, nby);
    return hipGetLastError();
}

bool fill_slots(SlotTab& S, const ViewTab* host_views, int a0, int a1, float src_y) {
    if (a1 - a0 > MAX_SLOTS) return false;
    for (int a = a0; a < a1; ++a) {
        const ViewTab& v = host_views[a];
        S.x0[a - a0] = v.x0;
        S.z0[a - a0] = v.z0;
        S.num[a - a0] = std::fma(v.z0, v.z0, std::fma(src_y, src_y, v.x0 * v.x0));
    }
    return true;
}

template <typename TP>
hipError_t sbp_t(const DevGeom& g, const SlotTab& S, int n, float* img, const void* prj,
                 hipStream_t st) {
    return by_sbp_rows<8>(g, SBP_ROWS_LINE, [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        hipLaunchKernelGGL((sbp_kernel<TP, R>), dim3(volume_tiles(g, R * CASE_WAVES)),
                           dim3(64 * CASE_WAVES), 0, st, g, S, n, (const TP*)prj, img);
        return hipGetLastError();
    });
}

template <int POT, typename TP, int R, int NW>
hipError_t batch_upd_t(const BatchCase* cases, const int* sched, int n_cases, int total, int grid,
                       int single_pass, hipStream_t st) {
    if (single_pass)
        hipLaunchKernelGGL((batch_update_kernel<POT, float, TP, R, NW, false>), dim3(grid),
                           dim3(64 * NW), 0, st, cases, sched, n_cases);
    else
        hipLaunchKernelGGL((batch_update_kernel<POT, float, TP, R, NW, true>), dim3(grid),
                           dim3(64 * NW), 0, st, cases, sched, n_cases);
    return hipGetLastError();
}

template <int POT, typename TP>
hipError_t batch_upd_s(int rows, int waves, const BatchCase* cases, const int* sched, int n_cases, int total,
                       int grid, int single, hipStream_t st) {
    if (rows == 8 && waves == 4) return batch_upd_t<POT, TP, 8, 4>(cases, sched, n_cases, total, grid, single, st);
    if (rows == 8 && waves == 2) return batch_upd_t<POT, TP, 8, 2>(cases, sched, n_cases, total, grid, single, st);
    if (rows == 4 && waves == 4) return batch_upd_t<POT, TP, 4, 4>(cases, sched, n_cases, total, grid, single, st);
    return hipErrorInvalidValue;
}

template <int POT>
hipError_t batch_upd_p(int prj_dtype, int rows, int waves, const BatchCase* cases,
                       const int* sched, int n_cases, int total, int grid, int single,
                       hipStream_t st) {
    switch (prj_dtype) {
        case OSTR_F32: return batch_upd_s<POT, float>(rows, waves, cases, sched, n_cases, total, grid, single, st);
        case OSTR_BF16: return batch_upd_s<POT, bf16_t>(rows, waves, cases, sched, n_cases, total, grid, single, st);
        case OSTR_F16: return batch_upd_s<POT, _Float16>(rows, waves, cases, sched, n_cases, total, grid, single, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool batch_update_shape_ok(int rows, int waves) {
    return (rows == 8 && (waves == 4 || waves == 2)) || (rows == 4 && waves == 4);
}

int64_t batch_upd_tiles(const DevGeom& g, int rows, int waves) {
    return volume_tiles(g, rows * waves);
}

void batch_slots(SlotTab& S, ViewTab* v, const ViewTab* host_views, int a0, int a1,
                 float src_y) {
    fill_slots(S, host_views, a0, a1, src_y);
    for (int a = a0; a < a1; ++a) v[a - a0] = host_views[a];
}

hipError_t launch_batch_update(const BatchCase* cases, const int* sched, int n_cases, int total, int grid,
                               int rows, int waves, int potential, int prj_dtype,
                               int single_pass, hipStream_t st) {
    if (total == 0) return hipSuccess;
    switch (potential) {
        case OSTR_PRIOR_Q2:
            return batch_upd_p<OSTR_PRIOR_Q2>(prj_dtype, rows, waves, cases, sched, n_cases, total, grid, single_pass, st);
        case OSTR_PRIOR_LANGE:
            return batch_upd_p<OSTR_PRIOR_LANGE>(prj_dtype, rows, waves, cases, sched, n_cases, total, grid, single_pass, st);
        case OSTR_PRIOR_HYPERBOLA:
            return batch_upd_p<OSTR_PRIOR_HYPERBOLA>(prj_dtype, rows, waves, cases, sched, n_cases, total, grid, single_pass, st);
    }
    return hipErrorInvalidValue;
}

size_t elem_size(int dtype) { return dtype == OSTR_F32 ? 4 : 2; }

hipError_t launch_transpose_bins(const void* src, void* dst, int n_slots, int nbx, int nby,
                                 int dtype, hipStream_t st) {
    if (n_slots <= 0) return hipSuccess;
    // 64x64 tiles write whole lines (9 views of 2048x1664 bins, FP32 35.7 us =
    // 6.9 TB/s through the caches, BF16 19.5; 32x32 tiles 36.4 and 28.6); below
    // 2 of them per CU 32x32 tiles, four times the groups (one view of 320x224:
    // 7.8 -> 4.6 us)
    const int64_t tiles = (int64_t)((nby + 63) / 64) * ((nbx + 63) / 64) * n_slots;
    const bool small = tiles < 512;
    if (dtype == OSTR_F32)
        return small ? transpose_t<float, 32>(src, dst, n_slots, nbx, nby, st)
                     : transpose_t<float, 64>(src, dst, n_slots, nbx, nby, st);
    return small ? transpose_t<uint16_t, 32>(src, dst, n_slots, nbx, nby, st)
                 : transpose_t<uint16_t, 64>(src, dst, n_slots, nbx, nby, st);
}

// `views` is the HOST copy of the slot table (slot parameters go to the kernel
// by value). prj is detector-row-major [slot][nby][nbx].
// The OS-SART updates carry a second sum per row and are faster at 4 rows than at
// 8 throughout (1000x500x45 voxels, 3 views, with the prior 179 and 204 us, without
// 86 and 88; 1400x600x60 389 and 423).
hipError_t launch_sart_update(const DevGeom& g, const ViewTab* views, int a0, int a1,
                              float* img, const float* diff_rows, const float* prior,
                              float lambda, float beta, hipStream_t st) {
    SlotTab S;
    if (!fill_slots(S, views, a0, a1, g.src_y)) return hipErrorInvalidValue;
    return by_sbp_rows<4>(g, SBP_ROWS_LINE, [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        const dim3 grid = group_grid(volume_tiles(g, R * CASE_WAVES), 64 * CASE_WAVES);
        const dim3 block(64 * CASE_WAVES);
        if (prior)
            hipLaunchKernelGGL((sart_update_kernel<float, true, R>), grid, block, 0, st, g, S,
                               a1 - a0, diff_rows, img, prior, lambda, beta);
        else
            hipLaunchKernelGGL((sart_update_kernel<float, false, R>), grid, block, 0, st, g,
                               S, a1 - a0, diff_rows, img, nullptr, lambda, 0.0f);
        return hipGetLastError();
    });
}

// 1400x600x60 voxels: 226 us at 8 rows per wave, 238 at 4 (256x256x48: 19.4 and 19.0)
hipError_t launch_huber_prior(const DevGeom& g, float* prior, const float* img, float delta,
                              hipStream_t st) {
    PriorW W27;
    prior_weights(W27.w, 1.0f);
    const PriorClass W = prior_params(W27, OSTR_PRIOR_HYPERBOLA, delta);
    return by_sbp_rows<8>(g, SBP_ROWS_LINE, [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        hipLaunchKernelGGL(huber_prior_kernel<R>, dim3(volume_tiles(g, R * CASE_WAVES)),
                           dim3(64 * CASE_WAVES), 0, st, g, W, 1.0f / delta, img, prior);
        return hipGetLastError();
    });
}

hipError_t launch_sart_update_fused(const DevGeom& g, const ViewTab* views, int a0, int a1,
                                    const float* x_in, float* x_out, const float* diff_rows,
                                    float lambda, float beta, float delta, hipStream_t st) {
    SlotTab S;
    if (!fill_slots(S, views, a0, a1, g.src_y)) return hipErrorInvalidValue;
    PriorW W27;
    prior_weights(W27.w, 1.0f);
    const PriorClass W = prior_params(W27, OSTR_PRIOR_HYPERBOLA, delta);
    return by_sbp_rows<4>(g, SBP_ROWS_LINE, [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        const dim3 grid = group_grid(volume_tiles(g, R * CASE_WAVES), 64 * CASE_WAVES);
        const dim3 block(64 * CASE_WAVES);
        if (beta != 0.0f)
            hipLaunchKernelGGL((sart_update_fused_kernel<true, R>), grid, block, 0, st, g, S,
                               a1 - a0, diff_rows, x_in, x_out, W, 1.0f / delta, lambda, beta);
        else
            hipLaunchKernelGGL((sart_update_fused_kernel<false, R>), grid, block, 0, st, g, S,
                               a1 - a0, diff_rows, x_in, x_out, W, 0.0f, lambda, 0.0f);
        return hipGetLastError();
    });
}

namespace {

UpdateCall update_call(const DevGeom& g, int n, const void* x_in, void* x_out, const float* d,
                       const void* hsub, int prj_dtype, float beta, float capl_scale,
                       int potential, float delta, float rho, int guard) {
    PriorW W27;
    prior_weights(W27.w, rho);
    return UpdateCall{g, n, x_in, x_out, d, hsub, prj_dtype, potential,
                      prior_params(W27, potential, delta),
                      potential == OSTR_PRIOR_Q2 ? 0.0f : 1.0f / delta, beta, capl_scale, guard};
}

}  // namespace

hipError_t launch_update_fused_matched(const DevGeom& g, const ViewTab* views, int a0, int a1,
                                       const void* x_in, void* x_out, int img_dtype,
                                       const float* d, const void* hsub, int prj_dtype,
                                       float beta, float capl_scale, int potential, float delta,
                                       float rho, int guard, hipStream_t st) {
    if (a1 - a0 > MAX_SLOTS || a1 < a0) return hipErrorInvalidValue;
    const MatchedSlots S = matched_slots(g, views + a0, a1 - a0);
    const UpdateCall u = update_call(g, a1 - a0, x_in, x_out, d, hsub, prj_dtype, beta,
                                     capl_scale, potential, delta, rho, guard);
    switch (img_dtype) {
        case OSTR_F32: return update_matched_f32(S, u, st);
        case OSTR_BF16: return update_matched_bf16(S, u, st);
        case OSTR_F16: return update_matched_f16(S, u, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_sbp_rows(const DevGeom& g, const ViewTab* views, int a0, int a1,
                           float* img_accum, const void* prj, int prj_dtype, hipStream_t st) {
    for (int b = a0; b < a1; b += MAX_SLOTS) {
        int e = b + MAX_SLOTS < a1 ? b + MAX_SLOTS : a1;
        SlotTab S;
        fill_slots(S, views, b, e, g.src_y);
        const int64_t off = (int64_t)(b - a0) * g.nbx * g.nby;
        hipError_t err;
        switch (prj_dtype) {
            case OSTR_F32:
                err = sbp_t<float>(g, S, e - b, img_accum, (const float*)prj + off, st);
                break;
            case OSTR_BF16:
                err = sbp_t<bf16_t>(g, S, e - b, img_accum, (const bf16_t*)prj + off, st);
                break;
            case OSTR_F16:
                err = sbp_t<_Float16>(g, S, e - b, img_accum, (const _Float16*)prj + off, st);
                break;
            default:
                return hipErrorInvalidValue;
        }
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}

hipError_t launch_update_fused(const DevGeom& g, const ViewTab* views, int a0, int a1,
                               const void* x_in, void* x_out, int img_dtype, const float* d,
                               const void* hsub, int prj_dtype, float beta, float capl_scale,
                               int potential, float delta, float rho, int guard,
                               hipStream_t st) {
    SlotTab S;
    if (!fill_slots(S, views, a0, a1, g.src_y)) return hipErrorInvalidValue;
    const UpdateCall u = update_call(g, a1 - a0, x_in, x_out, d, hsub, prj_dtype, beta,
                                     capl_scale, potential, delta, rho, guard);
    switch (img_dtype) {
        case OSTR_F32: return update_fused_f32(S, u, st);
        case OSTR_BF16: return update_fused_bf16(S, u, st);
        case OSTR_F16: return update_fused_f16(S, u, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace ostr
