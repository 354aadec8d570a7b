// Team kernels, BPTT with dL/d action_signal: see ring_team.hpp.
#include "ring_team_bptt.hpp"

// (dL/dA needs every product: several matrices in LDS gain 1 % from a kernel for their exact number)
hipError_t ring_launch_team_bptt_ga(const RingBpttArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  constexpr bool GA = true;
#define RING_TEAM_CASE(KPW, C16, MR, WK, FEW, MORE)                                                                   \
  if (sh.kpw == KPW && sh.c16 == C16 && sh.mr == MR && sh.wk == WK) {                                                 \
    if (sh.lds_mats == 0) RING_TEAM_RUN(KPW, C16, MR, WK, 0);                                                         \
    if constexpr (FEW >= 1) if (sh.lds_mats == 1) RING_TEAM_RUN(KPW, C16, MR, WK, 1);                                 \
    if constexpr (FEW >= 2 || MORE) RING_TEAM_RUN(KPW, C16, MR, WK, TEAM_MORE);                                                   \
  }
  RING_TEAM_SHAPES(RING_TEAM_CASE)
#undef RING_TEAM_CASE
  return hipErrorInvalidValue;
}
