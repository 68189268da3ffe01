// update_f16.hip - the fused OSTR updates (update_kernels.h) of FP16 images.
#include "update_kernels.h"

namespace ostr {

hipError_t update_fused_f16(const SlotTab& S, const UpdateCall& u, hipStream_t st) {
    return update_fused_image<_Float16>(S, u, st);
}
hipError_t update_matched_f16(const MatchedSlots& S, const UpdateCall& u, hipStream_t st) {
    return update_matched_image<_Float16>(S, u, st);
}

}  // namespace ostr
