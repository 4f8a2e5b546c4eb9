// Launchers of the split-row LR backward (attnres_lr_split.h), 16-byte vectors.
#include "attnres_lr_split.h"

namespace attnres {

template <class DT>
static hipError_t lr_split_bwd_dt(const ReadBwdParams& p, const Launch& L, hipStream_t st) {
  const dim3 g(L.grid), b(L.wpt * kWave);
#define ATTNRES_CASE16(NB)                                                                                    \
  case NB:                                                                                                    \
    if (L.teams == 1) hipLaunchKernelGGL((lr_split_bwd_kernel<DT, 16, NB, 1>), g, b, L.lds, st, p);           \
    else hipLaunchKernelGGL((lr_split_bwd_kernel<DT, 16, NB, 4>), g, b, L.lds, st, p);                        \
    return hipGetLastError();
  switch (L.nmax) { ATTNRES_LR_SPLIT_NB(ATTNRES_CASE16) }
#undef ATTNRES_CASE16
  return hipErrorInvalidValue;
}

hipError_t launch_lr_split_backward8(int dtype, const ReadBwdParams& p, const Launch& L, hipStream_t st);

hipError_t launch_lr_split_backward(int dtype, const ReadBwdParams& p, const Launch& L, hipStream_t st) {
  if (L.vb == 8) return launch_lr_split_backward8(dtype, p, L, st);
  ATTNRES_DISPATCH(dtype, lr_split_bwd_dt, p, L, st);
}

}  // namespace attnres
