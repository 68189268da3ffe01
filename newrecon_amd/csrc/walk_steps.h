// walk_steps.h - the Siddon walk's plain steps (device code of siddon.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ostr {

constexpr int WALK_BATCH = 4;  // walk steps per batch (two batches' gathers in flight)

// WALK_BATCH steps of a ray all of whose next steps are taken inside the
// volume: per step the segment (at - cur) len and the voxel's byte offset, then
// each axis whose next crossing is at `at` (ties: several) moves on by one
// voxel. Same operations as the flagged batch of walk(), without its flags.
// The moves run under the execution mask of their compare (v_cmpx), two adds
// per axis instead of two adds and two selects: 13 VALU instructions a step
// and one for the sum, against 26.5 with flags and selects. at and cur change
// roles every step (WALK_BATCH is even, so they end where they began). The
// read-write operands are early-clobber: the first step writes them, the later
// ones still read the inputs.
// What bounds the walk now is its gathers, not VALU issue: a wave's lanes stand
// in up to three slices and two rows, so a gather is 26-29 L1 accesses, and the
// L1 makes one per cycle and CU (texture data units busy 86% of the time, VALU
// issue 75%). A 3-view clinical subset (fproj_h) took 189 us with flagged batches
// only, 180 with this.
__device__ __forceinline__ void plain_steps(float& xn, float& yn, float& zn, uint32_t& px,
                                            uint32_t& py, uint32_t& pz, float& at, float& cur,
                                            float xi, float yi, float zi, uint32_t xs,
                                            uint32_t ys, uint32_t zs, float len,
                                            float (&seg)[WALK_BATCH],
                                            uint32_t (&off)[WALK_BATCH]) {
    static_assert(WALK_BATCH == 4, "the block below takes four steps");
    uint64_t lanes;
#define OSTR_STEP(AT, CUR, SEG, OFF)              \
    "v_sub_f32 " SEG ", " AT ", " CUR "\n"        \
    "v_add3_u32 " OFF ", %[px], %[py], %[pz]\n"   \
    "v_mul_f32 " SEG ", " SEG ", %[len]\n"        \
    "v_cmpx_eq_f32 vcc, " AT ", %[xn]\n"          \
    "v_add_f32 %[xn], %[xn], %[xi]\n"             \
    "v_add_u32 %[px], %[px], %[xs]\n"             \
    "s_mov_b64 exec, %[lanes]\n"                  \
    "v_cmpx_eq_f32 vcc, " AT ", %[yn]\n"          \
    "v_add_f32 %[yn], %[yn], %[yi]\n"             \
    "v_add_u32 %[py], %[py], %[ys]\n"             \
    "s_mov_b64 exec, %[lanes]\n"                  \
    "v_cmpx_eq_f32 vcc, " AT ", %[zn]\n"          \
    "v_add_f32 %[zn], %[zn], %[zi]\n"             \
    "v_add_u32 %[pz], %[pz], %[zs]\n"             \
    "s_mov_b64 exec, %[lanes]\n"                  \
    "v_min3_f32 " CUR ", %[xn], %[yn], %[zn]\n"
    asm volatile("s_mov_b64 %[lanes], exec\n"
                 OSTR_STEP("%[at]", "%[cur]", "%[s0]", "%[o0]")
                 OSTR_STEP("%[cur]", "%[at]", "%[s1]", "%[o1]")
                 OSTR_STEP("%[at]", "%[cur]", "%[s2]", "%[o2]")
                 OSTR_STEP("%[cur]", "%[at]", "%[s3]", "%[o3]")
                 : [xn] "+&v"(xn), [yn] "+&v"(yn), [zn] "+&v"(zn), [px] "+&v"(px), [py] "+&v"(py),
                   [pz] "+&v"(pz), [at] "+&v"(at), [cur] "+&v"(cur), [s0] "=&v"(seg[0]),
                   [s1] "=&v"(seg[1]), [s2] "=&v"(seg[2]), [s3] "=&v"(seg[3]),
                   [o0] "=&v"(off[0]), [o1] "=&v"(off[1]), [o2] "=&v"(off[2]),
                   [o3] "=&v"(off[3]), [lanes] "=&s"(lanes)
                 : [xi] "v"(xi), [yi] "v"(yi), [zi] "v"(zi), [xs] "v"(xs), [ys] "v"(ys),
                   [zs] "v"(zs), [len] "v"(len)
                 : "vcc");
#undef OSTR_STEP
}

}  // namespace ostr
