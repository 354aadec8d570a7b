// Team kernels, BPTT: see ring_team.hpp.
#include "ring_team_bptt.hpp"

hipError_t ring_launch_team_bptt(const RingBpttArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  constexpr bool GA = false;
#define RING_TEAM_CASE(KPW, C16, MR, WK, FEW, MORE)                                                                   \
  if (sh.kpw == KPW && sh.c16 == C16 && sh.mr == MR && sh.wk == WK) {                                                 \
    if (sh.lds_mats == 0) RING_TEAM_RUN(KPW, C16, MR, WK, 0);                                                         \
    if constexpr (FEW >= 1) if (sh.lds_mats == 1) RING_TEAM_RUN(KPW, C16, MR, WK, 1);                                 \
    if constexpr (FEW >= 2) if (sh.lds_mats == 2) RING_TEAM_RUN(KPW, C16, MR, WK, 2);                                 \
    if constexpr (FEW >= 3) if (sh.lds_mats == 3) RING_TEAM_RUN(KPW, C16, MR, WK, 3);                                 \
    if constexpr (FEW >= 4) if (sh.lds_mats == 4) RING_TEAM_RUN(KPW, C16, MR, WK, 4);                                 \
    if constexpr (MORE) RING_TEAM_RUN(KPW, C16, MR, WK, TEAM_MORE);                                                   \
  }
  RING_TEAM_SHAPES(RING_TEAM_CASE)
#undef RING_TEAM_CASE
  return hipErrorInvalidValue;
}
