// update_bf16.hip - the fused OSTR updates (update_kernels.h) of BF16 images.
#include "update_kernels.h"

namespace ostr {

hipError_t update_fused_bf16(const SlotTab& S, const UpdateCall& u, hipStream_t st) {
    return update_fused_image<bf16_t>(S, u, st);
}
hipError_t update_matched_bf16(const MatchedSlots& S, const UpdateCall& u, hipStream_t st) {
    return update_matched_image<bf16_t>(S, u, st);
}

}  // namespace ostr
