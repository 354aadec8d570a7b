// Team kernels, forward, two to four matrices in LDS: see ring_team_fwd.hpp.
#include "ring_team_fwd.hpp"

hipError_t ring_launch_team_fwd_lds4(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
#define RING_TEAM_CASE(KPW, C16, MR, WK, FEW, MORE)                                                 \
  if (sh.kpw == KPW && sh.c16 == C16 && sh.mr == MR && sh.wk == WK) {                               \
    if constexpr (FEW >= 2) if (sh.lds_mats == 2) { RING_TEAM_ACTS(KPW, C16, MR, WK, 2) }           \
    if constexpr (FEW >= 3) if (sh.lds_mats == 3) { RING_TEAM_ACTS(KPW, C16, MR, WK, 3) }           \
    if constexpr (FEW >= 4) if (sh.lds_mats == 4) { RING_TEAM_ACTS(KPW, C16, MR, WK, 4) }           \
  }
  RING_TEAM_SHAPES(RING_TEAM_CASE)
#undef RING_TEAM_CASE
  return hipErrorInvalidValue;
}
