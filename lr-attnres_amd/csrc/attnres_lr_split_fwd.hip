// Launchers of the split-row LR forward (attnres_lr_split.h).
#include "attnres_lr_split.h"

namespace attnres {

template <class DT>
static hipError_t lr_split_fwd_dt(const ReadParams& p, const Launch& L, hipStream_t st) {
  const dim3 g(L.grid), b(L.wpt * kWave);
#define ATTNRES_CASE16(NB) \
  case NB: hipLaunchKernelGGL((lr_split_fwd_kernel<DT, 16, NB>), g, b, L.lds, st, p); return hipGetLastError();
#define ATTNRES_CASE8(NB) \
  case NB: hipLaunchKernelGGL((lr_split_fwd_kernel<DT, 8, NB>), g, b, L.lds, st, p); return hipGetLastError();
  if (L.vb == 16) {
    switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE16) }
  } else if constexpr (sizeof(typename DT::S) == 2) {
    switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE8) ATTNRES_LR_SPLIT_NB8(ATTNRES_CASE8) }
  }
#undef ATTNRES_CASE16
#undef ATTNRES_CASE8
  return hipErrorInvalidValue;
}

hipError_t launch_lr_split_forward(int dtype, const ReadParams& p, const Launch& L, hipStream_t st) {
  ATTNRES_DISPATCH(dtype, lr_split_fwd_dt, p, L, st);
}

}  // namespace attnres
