// The matrix-core decodes under an attention mask: the formats' kernels with
// the mask compiled in, kept apart so that the plain ones keep their
// registers and schedule.
#include "decode_host.hpp"

namespace ss {

template <int D, class VF>
int launch_mfma_masked(const DecodeCommon &c, const typename VF::Args &va, const DecodeShape &s,
                       hipStream_t st, bool merge) {
    return launch_mfma_kernel<D, WithMask<VF>>(c, va, s, st, merge);
}

template <int NH8>
int launch_sunv_masked(const DecodeCommon &c, const typename VSunV<128, 4>::Args &va,
                       const DecodeShape &s, hipStream_t st) {
    return launch_sunv_mfma<NH8, true>(c, va, s, st);
}

#define SS_MASKED(DD, ...)                                                                      \
    template int launch_mfma_masked<DD, __VA_ARGS__>(                                           \
        const DecodeCommon &, const typename __VA_ARGS__::Args &, const DecodeShape &, hipStream_t, \
        bool);
#define SS_MASKED_GIL(DD, BB)        \
    SS_MASKED(DD, VGil<DD, BB, 1, float>)  \
    SS_MASKED(DD, VGil<DD, BB, 2, float>)  \
    SS_MASKED(DD, VGil<DD, BB, 1, __half>) \
    SS_MASKED(DD, VGil<DD, BB, 2, __half>)
SS_MASKED(128, VIl8Hyb<128>)
SS_MASKED(64, VIl8Hyb<64>)
SS_MASKED(128, VBf16<128>)
SS_MASKED(64, VBf16<64>)
SS_MASKED(128, VTq<128>)
SS_MASKED(64, VTq<64>)
SS_MASKED(128, VTqRows<128, 3>)
SS_MASKED(128, VTqRows<128, 4>)
SS_MASKED(64, VTqRows<64, 3>)
SS_MASKED(64, VTqRows<64, 4>)
SS_MASKED_GIL(128, 2)
SS_MASKED_GIL(128, 4)
SS_MASKED_GIL(64, 2)
SS_MASKED_GIL(64, 4)
#undef SS_MASKED_GIL
#undef SS_MASKED

#define SS_SUNV_MASKED(N)                                                                     \
    template int launch_sunv_masked<N>(const DecodeCommon &, const typename VSunV<128, 4>::Args &, \
                                       const DecodeShape &, hipStream_t);
SS_SUNV_MASKED(0)
SS_SUNV_MASKED(1)
SS_SUNV_MASKED(2)
SS_SUNV_MASKED(4)
SS_SUNV_MASKED(8)
#undef SS_SUNV_MASKED

}  // namespace ss
