// Launchers of the split-row LR backward (attnres_lr_split.h), 8-byte vectors (16-bit types).
#include "attnres_lr_split.h"

namespace attnres {

template <class DT>
static hipError_t lr_split_bwd8_dt(const ReadBwdParams& p, const Launch& L, hipStream_t st) {
  const dim3 g(L.grid), b(L.wpt * kWave);
#define ATTNRES_CASE8(NB)                                                                                     \
  case NB:                                                                                                    \
    if (L.teams == 1) hipLaunchKernelGGL((lr_split_bwd_kernel<DT, 8, NB, 1>), g, b, L.lds, st, p);            \
    else hipLaunchKernelGGL((lr_split_bwd_kernel<DT, 8, NB, 4>), g, b, L.lds, st, p);                         \
    return hipGetLastError();
  switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE8) ATTNRES_LR_SPLIT_NB8(ATTNRES_CASE8) }
#undef ATTNRES_CASE8
  return hipErrorInvalidValue;
}

hipError_t launch_lr_split_backward8(int dtype, const ReadBwdParams& p, const Launch& L, hipStream_t st) {
  if (dtype == ATTNRES_DTYPE_BF16) return lr_split_bwd8_dt<BF16>(p, L, st);
  if (dtype == ATTNRES_DTYPE_F16) return lr_split_bwd8_dt<F16>(p, L, st);
  return hipErrorInvalidValue;
}

}  // namespace attnres
