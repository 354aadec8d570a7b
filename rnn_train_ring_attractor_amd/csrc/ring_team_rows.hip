// Forward without a record over small teams for 128 < N <= 256 with two channels (protocol and pieces: ring_team.hpp),
// with the bits of the weight-resident forward (ring_res256.hip), so that a row comes out the same in any batch.
//
// That forward gives one compute unit the whole ring, 24 products for each of its 16 column tiles, and B = 1 pays the same
// step as B = 4096.  Here a member of a team has two column tiles and a compute wave the 24 products of one: it
// sums the whole contraction in the resident kernel's order, its K chunks first the even and then the odd ones, every
// matrix in an accumulator of its own, the gates afterwards.  One batch tile per team, so up to 32 tiles.
// us per call, T = 100, gelu: N = 256, B = 1: 142 -> 105; N = 256, B = 512: 137 -> 120; N = 200, B = 64: 142 -> 108.
// What bounds it is the hand-over's latency and the chain of 24 products (some 400 cycles).
#include "ring_team.hpp"

namespace {

constexpr int ROWS_TILES = 2, ROWS_CHUNKS = 8, ROWS_MATS = 3, ROWS_SLOTS = 8;

struct RowsOperand {
  u32x4 x[ROWS_CHUNKS];
  // (the memory clobber keeps a load from being folded into the same one a poll earlier)
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rsrc, const unsigned (&at)[ROWS_CHUNKS], unsigned base) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < ROWS_CHUNKS; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)at[i], (int)base, LD_COHERENT);
  }
  __device__ __forceinline__ bool ready() const {
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < ROWS_CHUNKS; ++i) m = max(max(m, max(x[i][0], x[i][1])), max(x[i][2], x[i][3]));
    return __ballot(m == EMPTY) == 0;
  }
};

}  // namespace

template <int ACT>
__global__ __launch_bounds__(64 * (ROWS_TILES + AUX)) void ring_team_rows_kernel(RingFwdArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  using TA = TeamAux<ROWS_TILES>;
  using AM = typename TA::AM;
  constexpr int NPT = TA::NPT;
  int team, mem;
  if (!team_coords(c, team, mem)) return;
  const LdsPlan L = lds_plan<ROWS_TILES, 1>(c.k, 1, 0, c.KC, 0, false, false);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const unsigned tile_bytes = (unsigned)c.KC * CHUNK_BYTES, slot_bytes = tile_bytes * (unsigned)c.nbt;
  const unsigned tile_at = (unsigned)team * tile_bytes;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  const int T = p.T;

  if (w < ROWS_TILES) {
    const int q = lane >> 4, b = lane & 15, out = 16 * (mem * ROWS_TILES + w) + b;
    unsigned at[ROWS_CHUNKS];
    bf16x8 wt[ROWS_MATS][ROWS_CHUNKS];
#pragma unroll
    for (int i = 0; i < ROWS_CHUNKS; ++i) {
      const int kc = rows_chunk(i);
      at[i] = kc < c.KC ? (unsigned)kc * CHUNK_BYTES + lane * 16 : NOWHERE;        // (past the contraction: zeros)
    }
    auto load = [&](auto how) {
      constexpr int HOW = decltype(how)::value, BATCH = HOW == WEIGHT_ROWS4 ? 8 : 4;
#pragma unroll
      for (int m = 0; m < ROWS_MATS; ++m)
#pragma unroll
        for (int i0 = 0; i0 < ROWS_CHUNKS; i0 += BATCH) {
          WeightLoad l[BATCH];
          const float* W = m == 0 ? c.Wo : c.Wa + (size_t)(m - 1) * c.N * c.N;
#pragma unroll
          for (int i = 0; i < BATCH; ++i) weight_load<HOW>(l[i], W, c.N, out, 32 * rows_chunk(i0 + i) + 8 * q);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < BATCH; ++i) {
            bf16x8 f = weight_fragment(l[i], c.N, out, 32 * rows_chunk(i0 + i) + 8 * q, m == 0 ? c.scale0 : 1.f, m == 0 ? c.shift0 : 0.f);
            asm volatile("" : "+v"(f));              // (here, not at its first use: twice the registers until then)
            wt[m][i0 + i] = f;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    };
    if ((c.N & 3) == 0) load(std::integral_constant<int, WEIGHT_ROWS4>{});
    else load(std::integral_constant<int, WEIGHT_ROWS>{});
    lds_barrier();                                        // the first gates are in LDS
    if (!team_go(lds, L)) return;
    float* const dst = share + w * AM::SHARE + q * AM::QS + b * 4;
    RowsOperand op;
    int slot = 0;
    bool dead = c.spin_max < 0;
    if (dead && lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
    op.issue(rsrc, at, tile_at);
    for (int t = 0; t < T; ++t) {
      const float* g = gl + (t & 1) * c.k * 16 + b;
      const float g1 = g[0], g2 = g[16];
      int spins = 0;
      while (!dead && !op.ready()) {
        if (++spins > c.spin_max) {
          dead = true;
          if (lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
        }
        op.issue(rsrc, at, (unsigned)slot * slot_bytes + tile_at);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0), for the compiler's books: this operand has landed on every path
      f32x4 P0 = {0.f, 0.f, 0.f, 0.f}, P1 = P0, P2 = P0;
#pragma unroll
      for (int i = 0; i < ROWS_CHUNKS; ++i) {
        const bf16x8 x = __builtin_bit_cast(bf16x8, op.x[i]);
        P1 = mfma16(wt[1][i], x, P1);
        P2 = mfma16(wt[2][i], x, P2);
        P0 = mfma16(wt[0][i], x, P0);
      }
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = fmaf(g2, P2[i], fmaf(g1, P1[i], P0[i]));
      *reinterpret_cast<f32x4*>(dst + (t & 1) * (ROWS_TILES * AM::SHARE)) = v;
      slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
      op.issue(rsrc, at, (unsigned)slot * slot_bytes + tile_at);      // (the first look at the next state)
      lds_barrier();
    }
    return;
  }

  __builtin_amdgcn_s_setprio(3);
  TA aux(c, mem, tid - 64 * ROWS_TILES);
  team_arrive(c, team, aux.at);
  const int N = p.N, B = p.B;
  const float oma = 1.f - p.alpha;
  const ActScale asc = act_scale_make(p.alpha);
  auto put = [&](int slot, unsigned x) { __builtin_amdgcn_raw_buffer_store_b32(x, rsrc, (int)aux.x_off, (int)((unsigned)slot * slot_bytes + tile_at), ST_LOCAL); };
  float r[NPT];
  aux.row_load(p.r_init, N, B, team, r);
  put(0, not_empty(pack_bf16(r[0], r[1])));
  const TeamGates tg(c, aux.at);
  auto gates_of = [&](int t) { return tg.fetch(c, t < T ? t : T - 1, team); };
  tg.put(gl, gates_of(0));
  float gA = gates_of(1), gB = gates_of(2);
  team_gather(c, lds, L, team, aux.at);
  lds_barrier();
  if (!team_go(lds, L)) return;

  int slot = 0, t = 0;
  auto step = [&](float& g) {
    tg.put(gl + ((t + 1) & 1) * c.k * 16, g);               // the next step's gates, fetched two steps ago
    lds_barrier();                                          // the step's products are complete
    float x[NPT], rn[NPT];
    aux.template sum_shares<1>(share, t & 1, x);
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      float aF, aD;
      act_scaled<ACT>(x[i], asc, aF, aD);
      rn[i] = aux.j0 + i < N ? fmaf(oma, r[i], aF) : 0.f;
    }
    const int next_slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
    put(next_slot, not_empty(pack_bf16(rn[0], rn[1])));     // (after the last step: nobody looks)
    g = gates_of(t + 3);
    put(slot == 0 ? ROWS_SLOTS - 1 : slot - 1, EMPTY);
    aux.row_store(p.hist + (size_t)t * B * N, N, B, team, rn);
#pragma unroll
    for (int i = 0; i < NPT; ++i) r[i] = rn[i];
    slot = next_slot;
    ++t;
  };
  while (t < T) {
    step(gA);
    if (t >= T) return;
    step(gB);
  }
}

RingTeamPlan ring_team_rows_plan(int N, int k, int B) {
  RingTeamPlan p{};
  if (!ring_res256_applicable(N, k)) return p;
  p.KC = (N + 31) / 32;
  p.G = (2 * p.KC + ROWS_TILES - 1) / ROWS_TILES;
  p.nteams = (B + 15) / 16;
  p.nt = 1;
  p.slots = ROWS_SLOTS;
  p.ok = p.nteams <= 8 * (32 / p.G);                       // (8 XCDs of 32 compute units)
  p.shape = RingTeamShape{ROWS_CHUNKS, ROWS_TILES, ROWS_MATS, ROWS_TILES, 0, 8 * p.G * ((p.nteams + 7) / 8)};
  p.xchg_bytes = (size_t)ROWS_SLOTS * p.nteams * p.KC * CHUNK_BYTES;
  p.gather_bytes = (size_t)p.nteams * RING_TEAM_WORD * sizeof(unsigned long long);
  return p;
}

hipError_t ring_launch_team_rows(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  const unsigned lds = lds_plan<ROWS_TILES, 1>(c.k, 1, 0, c.KC, 0, false, false).total;
  auto go = [&](auto kern) {
    return ring_team_start(reinterpret_cast<const void*>(kern), sh, c.G, lds, st,
                           [&](dim3 g, dim3 b, unsigned bytes) { RING_LAUNCH(kern, g, b, bytes, st, a, c); });
  };
  switch (a.act) {
    case ACT_RELU: return go(ring_team_rows_kernel<ACT_RELU>);
    case ACT_GELU: return go(ring_team_rows_kernel<ACT_GELU>);
    case ACT_TANH: return go(ring_team_rows_kernel<ACT_TANH>);
    case ACT_SILU: return go(ring_team_rows_kernel<ACT_SILU>);
    default: return hipErrorInvalidValue;
  }
}
