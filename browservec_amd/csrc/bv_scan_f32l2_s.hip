// Fused scan instantiations for codec C_F32L2_S (see bv_scan.h).
#include "bv_slots.h"

namespace bvk {

hipError_t scan_codec_f32l2_s(int lpr, int upl, const ScanArgs &a, uint32_t nq, hipStream_t s) {
    return dispatch_layout<C_F32L2_S>(Layout{lpr, upl}, a, nq, s);
}
hipError_t slots_codec_f32l2_s(int lpr, int upl, const SlotArgs &a, hipStream_t s) {
    return slots_layout<C_F32L2_S>(Layout{lpr, upl}, a, s);
}

}  // namespace bvk
