// update_kernels.h - the fused OSTR subset updates, with SBP and with the exact
// transpose, as templates over potential, storage types and rows per wave;
// update_f32.hip, update_bf16.hip and update_f16.hip instantiate them for one
// image storage type each.
#pragma once

#include "matched_device.h"
#include "sbp_device.h"

namespace ostr {

template <int POT, typename TI, typename TP, int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void update_fused_kernel(
    DevGeom g, SlotTab S, int n_slots, const TP* __restrict__ hsub, const TI* __restrict__ x_in,
    TI* __restrict__ x_out, const float* __restrict__ d, PriorClass W, float inv_delta,
    float beta, float capl_scale, int guard) {
    update_tile<POT, TI, TP, R, CASE_WAVES>(g, S, n_slots, hsub, x_in, x_out, d, W, inv_delta,
                                            beta, capl_scale, guard,
                                            xcd_tile(blockIdx.x, gridDim.x));
}

// Fused OSTR update with the exact transpose (the matched counterpart of
// update_fused_kernel): per voxel capL = M (0 + sum_views cos sum_i a_ij h_i)
// from matched_rows, then the prior window on x_in and the SQS update into
// x_out, the same epilogue (update_rows). h detector-row-major. R rows per
// lane (matched_row_count).
template <int POT, typename TI, typename TP, int R>
__global__ __launch_bounds__(64 * CASE_WAVES) void update_fused_matched_kernel(
    DevGeom g, MatchedSlots S, int n_slots, const TP* __restrict__ hsub,
    const TI* __restrict__ x_in, TI* __restrict__ x_out, const float* __restrict__ d,
    PriorClass W, float inv_delta, float beta, float capl_scale, int guard) {
    const TileCoord c = tile_coord<R, CASE_WAVES>(g, group_tile());
    if (c.iy0 >= g.ny || c.iz >= g.nz) return;  // see sbp_kernel
    const uint32_t nvox = (uint32_t)g.nx * g.ny * g.nz;
    const VolReader<TP> P(hsub, (uint32_t)n_slots * g.nbx * g.nby);
    const VolReader<TI> X(x_in, nvox);
    const VolWriter<TI> XO(x_out, nvox);
    const VolReader<float> D(d, nvox);
    float total[R];
    matched_rows<TP, R>(g, S, n_slots, 1, P, c.ix, c.iy0, c.iz, total);
    by_prior_mode<R>(g, c, W, [&](auto m) {
        update_rows<POT, decltype(m)::value, TI, R>(g, X, XO, D, c, total, W, inv_delta,
                                                    beta, capl_scale, guard);
    });
}

// f(potential, h type) as template arguments.
template <typename F>
hipError_t by_update_types(int potential, int prj_dtype, F f) {
    auto by_type = [&](auto pot) {
        switch (prj_dtype) {
            case OSTR_F32: return f(pot, (float*)nullptr);
            case OSTR_BF16: return f(pot, (bf16_t*)nullptr);
            case OSTR_F16: return f(pot, (_Float16*)nullptr);
        }
        return hipErrorInvalidValue;
    };
    switch (potential) {
        case OSTR_PRIOR_Q2: return by_type(std::integral_constant<int, OSTR_PRIOR_Q2>());
        case OSTR_PRIOR_LANGE: return by_type(std::integral_constant<int, OSTR_PRIOR_LANGE>());
        case OSTR_PRIOR_HYPERBOLA:
            return by_type(std::integral_constant<int, OSTR_PRIOR_HYPERBOLA>());
    }
    return hipErrorInvalidValue;
}

// 8 rows per wave from 120000 waves on for up to 3 views, where the window's loads
// weigh more: at 701x333x41 voxels (150183 waves) 4 and 8 rows take, us, one view
// and q2 47.3 and 44.8, Lange with BF16 h 71.7 and 69.7, hyperbola 66.9 and 67.8,
// but 9 views and q2 111.5 and 116.1.
template <typename TI>
hipError_t update_fused_image(const SlotTab& S, const UpdateCall& u, hipStream_t st) {
    return by_update_types(u.potential, u.prj_dtype, [&](auto pot, auto* h) {
        using TP = std::remove_pointer_t<decltype(h)>;
        return by_sbp_rows<8>(u.g, u.n_slots <= 3 ? 120000 : SBP_ROWS_LINE, [&](auto rows) {
            constexpr int R = decltype(rows)::value;
            hipLaunchKernelGGL((update_fused_kernel<decltype(pot)::value, TI, TP, R>),
                               dim3(volume_tiles(u.g, R * CASE_WAVES)), dim3(64 * CASE_WAVES), 0,
                               st, u.g, S, u.n_slots, (const TP*)u.hsub, (const TI*)u.x_in,
                               (TI*)u.x_out, u.d, u.W, u.inv_delta, u.beta, u.capl_scale,
                               u.guard);
            return hipGetLastError();
        });
    });
}

template <typename TI>
hipError_t update_matched_image(const MatchedSlots& S, const UpdateCall& u, hipStream_t st) {
    return by_update_types(u.potential, u.prj_dtype, [&](auto pot, auto* h) {
        using TP = std::remove_pointer_t<decltype(h)>;
        return by_matched_rows(u.g, [&](auto rows) {
            constexpr int R = decltype(rows)::value;
            hipLaunchKernelGGL((update_fused_matched_kernel<decltype(pot)::value, TI, TP, R>),
                               group_grid(volume_tiles(u.g, R * CASE_WAVES), 64 * CASE_WAVES),
                               dim3(64 * CASE_WAVES), 0, st, u.g, S, u.n_slots,
                               (const TP*)u.hsub, (const TI*)u.x_in,
                               (TI*)u.x_out, u.d, u.W, u.inv_delta, u.beta, u.capl_scale,
                               u.guard);
            return hipGetLastError();
        });
    });
}

}  // namespace ostr
