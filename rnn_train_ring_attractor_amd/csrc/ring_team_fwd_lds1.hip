// Team kernels, forward, one matrix in LDS: see ring_team_fwd.hpp.
#include "ring_team_fwd.hpp"

hipError_t ring_launch_team_fwd_lds1(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
#define RING_TEAM_CASE(KPW, C16, MR, WK, FEW, MORE)                                                 \
  if (sh.kpw == KPW && sh.c16 == C16 && sh.mr == MR && sh.wk == WK) {                               \
    if constexpr (FEW >= 1) if (sh.lds_mats == 1) { RING_TEAM_ACTS(KPW, C16, MR, WK, 1) }           \
  }
  RING_TEAM_SHAPES(RING_TEAM_CASE)
#undef RING_TEAM_CASE
  return hipErrorInvalidValue;
}
