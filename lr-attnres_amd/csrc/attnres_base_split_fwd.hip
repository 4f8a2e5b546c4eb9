// Launchers of the split-row base forward (attnres_base_split.h).
#include "attnres_base_split.h"

namespace attnres {

// L.vb = vector bytes (8: 16-bit types only), L.nmax = source slots
template <class DT>
static hipError_t base_split_fwd_dt(const ReadParams& p, const Launch& L, hipStream_t st) {
  const dim3 g(L.grid), b(L.wpt * kWave);
#define ATTNRES_CASE16(NB) \
  case NB: hipLaunchKernelGGL((base_split_fwd_kernel<DT, 16, NB>), g, b, 0, st, p); return hipGetLastError();
#define ATTNRES_CASE8(NB) \
  case NB: hipLaunchKernelGGL((base_split_fwd_kernel<DT, 8, NB>), g, b, 0, st, p); return hipGetLastError();
  if (L.vb == 16) {
    switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE16) }
  } else if constexpr (sizeof(typename DT::S) == 2) {
    switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE8) ATTNRES_LR_SPLIT_NB8(ATTNRES_CASE8) }
  }
#undef ATTNRES_CASE16
#undef ATTNRES_CASE8
  return hipErrorInvalidValue;
}

hipError_t launch_base_split_forward(int dtype, const ReadParams& p, const Launch& L, hipStream_t st) {
  ATTNRES_DISPATCH(dtype, base_split_fwd_dt, p, L, st);
}

}  // namespace attnres
