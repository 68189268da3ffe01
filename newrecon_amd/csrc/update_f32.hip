// update_f32.hip - the fused OSTR updates (update_kernels.h) of FP32 images.
#include "update_kernels.h"

namespace ostr {

hipError_t update_fused_f32(const SlotTab& S, const UpdateCall& u, hipStream_t st) {
    return update_fused_image<float>(S, u, st);
}
hipError_t update_matched_f32(const MatchedSlots& S, const UpdateCall& u, hipStream_t st) {
    return update_matched_image<float>(S, u, st);
}

}  // namespace ostr
