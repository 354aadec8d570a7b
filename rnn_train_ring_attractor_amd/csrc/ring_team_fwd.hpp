// Team kernels, forward: see ring_team.hpp.  (Sources by how many matrices are in LDS: one, two to four, any number or none.)
#pragma once
#include "ring_team.hpp"

// ------------------------------------------------------------------------------------------------
// Forward.  p.dfrag / p.rfrag may be null together (inference).
// ------------------------------------------------------------------------------------------------
template <int KPW, int C16, int MR, int WK, int EX, int ACT, bool LATE>
__global__ __launch_bounds__(64 * (WK + AUX)) void ring_team_fwd_kernel(RingFwdArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int team, mem;
  if (!team_coords(c, team, mem)) return;
  const LdsPlan L = lds_plan<C16, WK>(c.k, c.nt, EX ? c.k + 1 - MR : 0, c.KC, parked_bytes(KPW, C16, MR, WK), false, false);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int my_nt = (c.nbt - team + c.nteams - 1) / c.nteams;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const int T = p.T;

  if (w < WK) {
    team_compute_loop<false, KPW, C16, MR, WK, EX, false, LATE>(c, L, lds, rsrc, mem, team, my_nt, T, w, lane);
    return;
  }

  __builtin_amdgcn_s_setprio(3);       // the epilogue is the serial part: its wave goes first on the SIMD it shares with two others
  using TA = TeamAux<C16>;
  constexpr int NPT = TA::NPT;
  TA aux(c, mem, tid - 64 * WK);
  team_arrive(c, team, aux.at);
  const int at = aux.at, N = p.N, B = p.B, nbt = p.nbt;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const state = reinterpret_cast<float*>(lds + L.state) + at * NPT;
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  const float oma = 1.f - p.alpha;
  const ActScale asc = act_scale_make(p.alpha);
  const bool save = p.dfrag != nullptr;

  for (int j = 0; j < my_nt; ++j) {
    const int bt = team + c.nteams * j;
    float r[NPT];
    aux.row_load(p.r_init, N, B, bt, r);
    if (aux.map.active) {
#pragma unroll
      for (int i = 0; i < NPT; ++i) state[(size_t)j * C16 * 256 + i] = r[i];
    }
    aux.publish(c, rsrc, 0, bt, r);
  }
  const TeamGates tg(c, at);
  auto gates_of = [&](const ItemCursor& cu) { return tg.fetch(c, cu.s, team + c.nteams * cu.j); };
  ItemCursor cur{0, 0};
  tg.put(gl, gates_of(cur));
  cur.advance(my_nt, T);
  float gA = gates_of(cur);               // items 1 and 2
  cur.advance(my_nt, T);
  float gB = gates_of(cur);
  team_gather(c, lds, L, team, at);
  lds_barrier();
  if (!team_go(lds, L)) return;

  int slot = 0, it = 0, t = 0, j = 0;
  bool done = false;
  auto item = [&](float& g) {
    const int next_slot = slot + 1 == c.slots ? 0 : slot + 1;
    const int bt = team + c.nteams * j;
    float r[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) r[i] = state[(size_t)j * C16 * 256 + i];
    tg.put(gl + ((it + 1) & 1) * c.k * 16, g);              // the next item's gates, fetched two items ago
    lds_barrier();                                          // the item's shares are complete
    float x[NPT], aF[NPT], rn[NPT];
    ActRecord<ACT> rd[NPT];
    aux.template sum_shares<WK>(share, it & 1, x);
#pragma unroll
    for (int i = 0; i < NPT; ++i) aF[i] = rd[i].apply(x[i], asc);
    // Rows past B need no mask: their operand, row sum and initial state are zero and every F(0) is zero.  Neurons past N
    // see the J0 term.
#pragma unroll
    for (int i = 0; i < NPT; ++i) rn[i] = aux.j0 + i < N ? fmaf(oma, r[i], aF[i]) : 0.f;
    aux.publish(c, rsrc, next_slot, bt, rn);                // (after the last step: nobody looks)
    cur.advance(my_nt, T);
    g = gates_of(cur);                                      // item it + 3
    if (aux.map.active) {
#pragma unroll
      for (int i = 0; i < NPT; ++i) state[(size_t)j * C16 * 256 + i] = rn[i];
    }
    aux.refill(c, rsrc, slot == 0 ? c.slots - 1 : slot - 1, bt);
    aux.row_store(p.hist + (size_t)t * B * N, N, B, bt, rn);
    unsigned d[NPT / 2];
#pragma unroll
    for (int i = 0; i < NPT / 2; ++i) d[i] = ActRecord<ACT>::pair_once(asc, rd[2 * i], rd[2 * i + 1]);
    aux.dact_store(p.dfrag, t, nbt, bt, c.cts, d);
    if (save && (t & 1) == 0) {        // this step's operand and the next one's are both in hand: one 16-byte slot
      unsigned lo[NPT / 2], hi[NPT / 2];
#pragma unroll
      for (int i = 0; i < NPT / 2; ++i) {
        lo[i] = pack_bf16(r[2 * i], r[2 * i + 1]);
        hi[i] = t + 1 < T ? pack_bf16(rn[2 * i], rn[2 * i + 1]) : 0u;
      }
      aux.pair_put(p.rfrag, t, nbt, bt, c.cts, lo, hi);
    }
    ++it;
    if (++j == my_nt) {
      j = 0;
      slot = next_slot;
      done = ++t >= T;
    }
  };
  while (!done) {
    item(gA);
    if (done) return;
    item(gB);
  }
}

template <int KPW, int C16, int MR, int WK, int EX, int ACT, bool LATE>
hipError_t team_fwd_start(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  auto kern = ring_team_fwd_kernel<KPW, C16, MR, WK, EX, ACT, LATE>;
  return ring_team_start(reinterpret_cast<const void*>(kern), sh, c.G,
                         lds_plan<C16, WK>(c.k, c.nt, sh.lds_mats, c.KC, parked_bytes(KPW, C16, MR, WK), false, false).total, st,
                         [&](dim3 g, dim3 b, unsigned lds) { RING_LAUNCH(kern, g, b, lds, st, a, c); });
}
#define RING_TEAM_ACT(KPW, C16, MR, WK, EX, ACT)                                                                    \
  if constexpr (team_may_look_late(KPW, C16, MR, WK, EX))                                                           \
    if (c.look >= 0) return team_fwd_start<KPW, C16, MR, WK, EX, ACT, true>(a, c, sh, st);                          \
  return team_fwd_start<KPW, C16, MR, WK, EX, ACT, false>(a, c, sh, st)
#define RING_TEAM_ACTS(KPW, C16, MR, WK, EX)                                  \
  switch (a.act) {                                                            \
    case ACT_RELU: RING_TEAM_ACT(KPW, C16, MR, WK, EX, ACT_RELU);             \
    case ACT_GELU: RING_TEAM_ACT(KPW, C16, MR, WK, EX, ACT_GELU);             \
    case ACT_TANH: RING_TEAM_ACT(KPW, C16, MR, WK, EX, ACT_TANH);             \
    case ACT_SILU: RING_TEAM_ACT(KPW, C16, MR, WK, EX, ACT_SILU);             \
    default: return hipErrorInvalidValue;                                     \
  }
