// Dispatch of the block-sparse forward to the translation unit that holds the kernels for the element type,
// for the source of the PARTIAL tiles' mask entries and for the way Q tiles are handed out (sparse_fwd_inst.hip).
#include "kernels.h"

namespace sa {

template <int DT, bool PK, int HOW>
hipError_t launch_fwd_variant(const FwdParams &p, int D, int BQ, hipStream_t stream);
#define SA_DECL(DT, PK, HOW) \
    extern template hipError_t launch_fwd_variant<DT, PK, HOW>(const FwdParams &, int, int, hipStream_t);
SA_DECL(0, false, 0) SA_DECL(0, false, 1) SA_DECL(0, false, 2) SA_DECL(0, true, 0) SA_DECL(0, true, 1) SA_DECL(0, true, 2)
SA_DECL(0, true, 3) SA_DECL(1, true, 3)
SA_DECL(0, false, 4) SA_DECL(0, true, 4) SA_DECL(1, false, 4) SA_DECL(1, true, 4)
SA_DECL(0, false, 5) SA_DECL(0, true, 5) SA_DECL(1, false, 5) SA_DECL(1, true, 5)
SA_DECL(1, false, 0) SA_DECL(1, false, 1) SA_DECL(1, false, 2) SA_DECL(1, true, 0) SA_DECL(1, true, 1) SA_DECL(1, true, 2)
#undef SA_DECL

namespace {
template <int DT, bool PK>
hipError_t by_hand_out(const FwdParams &p, int D, int BQ, hipStream_t stream) {
    if (p.sched != nullptr) return launch_fwd_variant<DT, PK, 1>(p, D, BQ, stream);
    if (p.ragged) {
        if constexpr (PK) return launch_fwd_variant<DT, PK, 3>(p, D, BQ, stream);
        else return hipErrorInvalidValue;
    }
    if (p.halves) return launch_fwd_variant<DT, PK, 4>(p, D, BQ, stream);
    if (p.nsplit <= 1) return launch_fwd_variant<DT, PK, 0>(p, D, BQ, stream);
    if (p.split_chunks == 0) return p.tag != 0 ? launch_fwd_variant<DT, PK, 5>(p, D, BQ, stream) : hipErrorInvalidValue;
    const hipError_t e = launch_fwd_variant<DT, PK, 2>(p, D, BQ, stream);
    return e != hipSuccess || p.tag != 0 ? e : launch_fwd_merge(p, DT, D, BQ, stream);
}
}  // namespace

hipError_t launch_fwd(const FwdParams &p, int dtype, int D, int BQ, hipStream_t stream) {
    const bool pk = p.packed != nullptr;
    if (dtype == 0) return pk ? by_hand_out<0, true>(p, D, BQ, stream) : by_hand_out<0, false>(p, D, BQ, stream);
    if (dtype == 1) return pk ? by_hand_out<1, true>(p, D, BQ, stream) : by_hand_out<1, false>(p, D, BQ, stream);
    return hipErrorInvalidValue;
}

}  // namespace sa
