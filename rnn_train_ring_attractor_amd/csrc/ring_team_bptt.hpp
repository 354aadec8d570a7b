// The team BPTT kernel; instantiated in ring_team_bptt.hip and ring_team_bptt_ga.hip.
#pragma once
#include "ring_team.hpp"

// ------------------------------------------------------------------------------------------------
// BPTT, reverse time.  Operand number s is g of step T - 1 - s; the products of round s give the carry into step
// T - 2 - s (the last round, which only grad_r_init needs, is left out when that is not asked for).
// ------------------------------------------------------------------------------------------------
template <int KPW, int C16, int MR, int WK, int EX, bool GA, bool LATE>
__global__ __launch_bounds__(64 * (WK + AUX)) void ring_team_bptt_kernel(RingBpttArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int team, mem;
  if (!team_coords(c, team, mem)) return;
  const LdsPlan L = lds_plan<C16, WK>(c.k, c.nt, EX ? c.k + 1 - MR : 0, c.KC, parked_bytes(KPW, C16, MR, WK), true, GA);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int my_nt = (c.nbt - team + c.nteams - 1) / c.nteams;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const int T = p.T;
  const int steps = (p.grad_r_init || GA) ? T : T - 1;

  if (w < WK) {
    team_compute_loop<true, KPW, C16, MR, WK, EX, GA, LATE>(c, L, lds, rsrc, mem, team, my_nt, steps, w, lane);
    return;
  }

  __builtin_amdgcn_s_setprio(3);       // the epilogue is the serial part: its wave goes first on the SIMD it shares with two others
  using TA = TeamAux<C16>;
  constexpr int NPT = TA::NPT;
  TA aux(c, mem, tid - 64 * WK);
  team_arrive(c, team, aux.at);
  const int at = aux.at, N = p.N, B = p.B, nbt = p.nbt;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const state = reinterpret_cast<float*>(lds + L.state) + at * NPT;         // (1 - alpha) G
  unsigned* const held = reinterpret_cast<unsigned*>(lds + L.held) + at * (NPT / 2);   // bf16 g of an odd step
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  float* const rows = reinterpret_cast<float*>(lds + L.rows);
  const float* const ga = reinterpret_cast<const float*>(lds + L.ga);
  const float oma = 1.f - p.alpha;
  const bool loss = p.loss_coef != nullptr;
  const TeamGates tg(c, at);
  float cs[NPT], sn[NPT], up = 0.f;
#pragma unroll
  for (int i = 0; i < NPT; ++i) { cs[i] = 0.f; sn[i] = 0.f; }
  if (loss) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const float phi = 6.2831853071795864769f * (float)(aux.j0 + i) / (float)N;
      cs[i] = cosf(phi);
      sn[i] = sinf(phi);
    }
    up = (p.loss_upstream ? p.loss_upstream[0] : 1.f) * p.loss_inv_rows;
  }

  const char* const coef = loss ? reinterpret_cast<const char*>(p.loss_coef) : reinterpret_cast<const char*>(c.Wo);
  struct In {
    float go[NPT];
    _Float16 d[NPT];
    f32x3 cf;
    float rp[GA ? NPT : 1];
    float g;
  };
  // what the epilogue of round s (it forms g of step T - 2 - s) needs; and the gates of the products' step
  auto fetch = [&](const ItemCursor& cu, In& in) {
    const int bt = team + c.nteams * cu.j;
    const int t = T - 2 - cu.s < 0 ? 0 : T - 2 - cu.s;
    aux.row_load_raw((loss ? p.hist : p.grad_out) + (size_t)t * B * N, N, B, bt, in.go);
    const _Float16* src = p.dfrag + aux.dact_offset(t, nbt, bt, c.cts);
    if constexpr (NPT == 4) {
      const f16x4 v = *reinterpret_cast<const f16x4*>(src);
#pragma unroll
      for (int i = 0; i < 4; ++i) in.d[i] = v[i];
    } else {
      const f16x2 v = *reinterpret_cast<const f16x2*>(src);
      in.d[0] = v[0];
      in.d[1] = v[1];
    }
    const int b = 16 * bt + aux.map.b;
    in.cf = *reinterpret_cast<const f32x3*>(coef + (loss ? ((size_t)t * B + (b < B ? b : B - 1)) * 16 : 0));   // (without the loss head: any 16 bytes, unused)
  };
  // the gates of round s's products belong to step T - 1 - s; with dL/dA also r_prev of that step
  auto fetch_side = [&](const ItemCursor& cu, In& in) {
    const int bt = team + c.nteams * cu.j, t = T - 1 - cu.s < 0 ? 0 : T - 1 - cu.s;
    in.g = tg.fetch(c, t, bt);
    if constexpr (GA) {
      float v[NPT];
      aux.row_load_raw(t == 0 ? p.r_init : p.hist + (size_t)(t - 1) * B * N, N, B, bt, v);
#pragma unroll
      for (int i = 0; i < NPT; ++i) in.rp[i] = v[i];
    }
  };
  auto put_side = [&](int buf, const In& in) {
    tg.put(gl + buf * c.k * 16, in.g);
    if constexpr (GA) {
      if (aux.map.active) {
        float v[NPT];
#pragma unroll
        for (int i = 0; i < NPT; ++i) v[i] = in.rp[i];
        aux.align(N, v);
        float* dst = rows + buf * C16 * 256 + aux.map.c * 256 + (aux.map.q * 16 + aux.map.b) * 4 + 2 * aux.map.p;
#pragma unroll
        for (int i = 0; i < NPT; ++i) dst[i] = v[i];
      }
    }
  };
  // carry in -> G, g of the step, and g's bf16 pairs
  auto form_g = [&](const In& in, const float (&carry)[NPT], int bt, float (&G)[NPT], float (&gg)[NPT], unsigned (&x)[NPT / 2]) {
    const bool rowok = 16 * bt + aux.map.b < B;
    float gin[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) gin[i] = in.go[i];
    aux.align(N, gin);
    float kc = 0.f, ks = 0.f, beta = 0.f;
    if (loss) {
      kc = in.cf[0] * up;
      ks = in.cf[1] * up;
      beta = in.cf[2] * up;
    }
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      float go = gin[i];
      if (loss) {
        const float r = go;
        go = fmaf(kc, cs[i], fmaf(ks, sn[i], r > 0.f ? beta : (r < 0.f ? -beta : 0.f)));
      }
      const bool ok = rowok && aux.j0 + i < N;
      G[i] = ok ? go + carry[i] : 0.f;
      gg[i] = ok ? (float)in.d[i] * G[i] : 0.f;      // the record carries alpha
    }
#pragma unroll
    for (int i = 0; i < NPT / 2; ++i) x[i] = pack_bf16(gg[2 * i], gg[2 * i + 1]);
  };
  // (1 - alpha) G for the next round; the copy for the weight gradients, a pair of steps at a time
  auto keep_g = [&](const float (&G)[NPT], const unsigned (&x)[NPT / 2], int t, int j) {
    unsigned* h = held + (size_t)j * C16 * 128;
    if (aux.map.active) {
#pragma unroll
      for (int i = 0; i < NPT; ++i) state[(size_t)j * C16 * 256 + i] = oma * G[i];
    }
    if (t & 1) {
      if (aux.map.active) {
#pragma unroll
        for (int i = 0; i < NPT / 2; ++i) h[i] = x[i];
      }
    } else {
      unsigned hi[NPT / 2];
#pragma unroll
      for (int i = 0; i < NPT / 2; ++i) hi[i] = t + 1 < T && aux.map.active ? h[i] : 0u;
      aux.pair_put(p.gfrag, t, nbt, team + c.nteams * j, c.cts, x, hi);
    }
  };
  auto flush_ga = [&](int s, int j, int buf) {       // sums the waves' shares in wave order; one partial per member
    if constexpr (GA) {
      const int bt = team + c.nteams * j, t = T - 1 - s;
      for (int idx = at; idx < 16 * c.k; idx += 256) {
        const int ch = idx >> 4, row = idx & 15, b = 16 * bt + row;
        const float* src = ga + ((size_t)buf * WK * c.k + ch) * 16 + row;
        float v = 0.f;
#pragma unroll
        for (int x = 0; x < WK; ++x) v += src[(size_t)x * c.k * 16];
        if (b < B) c.ga_part[(((size_t)mem * T + t) * c.k + ch) * B + b] = v;
      }
    }
  };

  // operand 0: g of step T - 1, no carry yet
  for (int j = 0; j < my_nt; ++j) {
    In in;
    ItemCursor cu{-1, j};
    fetch(cu, in);
    float zero[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) zero[i] = 0.f;
    float G[NPT], gg[NPT];
    unsigned x[NPT / 2];
    form_g(in, zero, team + c.nteams * j, G, gg, x);
    aux.publish(c, rsrc, 0, team + c.nteams * j, gg);
    keep_g(G, x, T - 1, j);
  }
  if (steps == 0) {
    team_gather(c, lds, L, team, at);
    lds_barrier();
    return;
  }
  // Register set A serves the even items, B the odd ones.  At item `it` a set holds that item's grad_output and
  // derivative record, and the gates (and r_prev rows) of item it + 1, all fetched two items earlier.
  In inA, inB;
  ItemCursor near{0, 0}, far{0, 0};
  fetch_side(far, inA);
  put_side(0, inA);
  far.advance(my_nt, steps);
  fetch(near, inA);
  fetch_side(far, inA);
  near.advance(my_nt, steps);
  far.advance(my_nt, steps);
  fetch(near, inB);
  fetch_side(far, inB);
  team_gather(c, lds, L, team, at);
  lds_barrier();
  if (!team_go(lds, L)) return;

  int slot = 0, it = 0, s = 0, j = 0;
  bool done = false;
  auto item = [&](In& in) {
    const int bt = team + c.nteams * j;
    const int next_slot = slot + 1 == c.slots ? 0 : slot + 1;
    float carry[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) carry[i] = state[(size_t)j * C16 * 256 + i];
    put_side((it + 1) & 1, in);                      // gates (and r_prev rows) of the next item
    lds_barrier();
    float x[NPT], G[NPT], gg[NPT];
    unsigned pk[NPT / 2];
    aux.template sum_shares<WK>(share, it & 1, x);
#pragma unroll
    for (int i = 0; i < NPT; ++i) carry[i] += x[i];
    form_g(in, carry, bt, G, gg, pk);
    aux.publish(c, rsrc, next_slot, bt, gg);           // (after the last round: nobody looks)
    near.advance(my_nt, steps);
    far.advance(my_nt, steps);
    fetch(near, in);                                   // item it + 2
    fetch_side(far, in);                               // item it + 3
    aux.refill(c, rsrc, slot == 0 ? c.slots - 1 : slot - 1, bt);
    if (s + 1 < T) {
      keep_g(G, pk, T - 2 - s, j);
    } else if (p.grad_r_init) {
      // masked like g: rows past B and neurons past N are not stored
      aux.row_store(p.grad_r_init, N, B, bt, carry);
    }
    flush_ga(s, j, it & 1);
    ++it;
    if (++j == my_nt) {
      j = 0;
      ++s;
      slot = next_slot;
    }
    done = s >= steps;
  };
  while (!done) {
    item(inA);
    if (done) break;
    item(inB);
  }
}

template <int KPW, int C16, int MR, int WK, int EX, bool GA, bool LATE>
hipError_t team_bptt_start(const RingBpttArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  auto kern = ring_team_bptt_kernel<KPW, C16, MR, WK, EX, GA, LATE>;
  return ring_team_start(reinterpret_cast<const void*>(kern), sh, c.G,
                         lds_plan<C16, WK>(c.k, c.nt, sh.lds_mats, c.KC, parked_bytes(KPW, C16, MR, WK), true, GA).total, st,
                         [&](dim3 g, dim3 b, unsigned lds) { RING_LAUNCH(kern, g, b, lds, st, a, c); });
}
#define RING_TEAM_RUN(KPW, C16, MR, WK, EX)                                                                           \
  do {                                                                                                                \
    if constexpr (team_may_look_late(KPW, C16, MR, WK, EX))                                                           \
      if (c.look >= 0) return team_bptt_start<KPW, C16, MR, WK, EX, GA, true>(a, c, sh, st);                          \
    return team_bptt_start<KPW, C16, MR, WK, EX, GA, false>(a, c, sh, st);                                            \
  } while (0)
