// Time loops over small teams for 128 < N <= 256 with two channels (protocol and pieces: ring_team.hpp), with the bits and
// the record of the weight-resident kernels (ring_res256.hip), so that a row comes out the same in any batch and either
// family's backward reads either one's record.
//
// Those kernels give one compute unit the whole ring, 24 products for each of its 16 column tiles, and B = 1 pays the same
// step as B = 4096.  Here a member of a team has one column tile and a compute wave for the eight products of each matrix, or
// two and one for all 24 of each (RowsSplit).  A wave sums the whole contraction in the resident kernel's order (forward: its
// K chunks first the even and then the odd ones; BPTT: one after the other, the ungated sum starting from (1 - alpha) G), every
// matrix in an accumulator of its own, the gates afterwards.  One batch tile per team, so up to 32 tiles.
// us per call, T = 100, weight-resident kernels -> here with two column tiles and before team_look -> now with one.  With a record:
// N = 256, B = 128, gelu: forward 143 -> 117 -> 100, BPTT 138 -> 130 -> 113; N = 200, B = 64: 156 -> 110 and 245 -> 120; N = 256,
// B = 128, relu, with the loss's gradient and dL/dA: 165 -> 114 (its row sums by a pass of their own included) and 222 -> 149.
// Without: N = 256, B = 1: 142 -> 99 -> 80.
// What bounds it is the hand-over's latency, a chain of eight products (24 with two tiles, some 400 cycles) and the sums and the
// activation behind a barrier, one after the other.
#include "ring_team.hpp"

namespace {

constexpr int ROWS_CHUNKS = 8, ROWS_MATS = 3, ROWS_SLOTS = 8;
// Two column tiles a member and a compute wave for the 24 products of each, or one column tile and a compute wave for the eight of
// each matrix (the gates then follow in the auxiliary waves, in the same order): the chain a step waits for is 250 cycles shorter, but
// takes twice the compute units and half as much more of the operand into each.  us a call, T = 100, two and one, before team_look:
// forward N = 256, B = 16, relu 96.3 and 86.6, tanh 99.2 and 94.1, B = 1, gelu 93.2 and 90.9, B = 256, gelu 105.2 and 103.8; training
// N = 200, B = 64, tanh 245 and 232.  So one where members of one find room for every batch tile (256 rows; 384 at N <= 160 without a
// record, where a team has ten members instead of sixteen), beside as many launches as are under way on other streams: two tiles let
// twice as many of them run at once.  Under capture, where nobody knows what a graph will be replayed beside, as if there were one
// other.  us a call, gelu, T = 100, always one tile, always two, and so:
//   eager, streams         1                    2                    3                    4
//     N = 256, B = 1      83.6   94.0   83.6   45.5   50.3   45.4   70.0   34.1   34.2   74.9   33.0   32.6
//     N = 256, B = 128    93.6  102.6   94.0   51.3   55.0   51.2  103.5   38.0   38.1  109.2   55.0   55.4
//     N = 256, B = 200    95.5  103.2   95.9   93.8   56.1   55.9  105.6   52.4   52.3  110.7   50.7   50.9
//   graphs, replayed on a stream each (B = 200: four that want all compute units starve each other until they give up)
//     N = 256, B = 128   101.4  109.5  101.2   53.1   56.7   52.7   49.4   39.3   49.4   46.3   37.8   48.9
//     N = 256, B = 200   103.5  111.3  110.9   96.8   57.2   57.2   99.0   75.0   75.1   2659   52.7   52.8
template <int TILES>
struct RowsSplit {
  static constexpr int SHARES = TILES == 1 ? ROWS_MATS : 1, WAVES = TILES * SHARES;     // shares of a column tile, compute waves
  // (the plan has room for the dL/dA shares of one column tile a share, behind everything else)
  static constexpr unsigned GA_MORE = 2 * 2 * (TILES - 1) * 16 * sizeof(float);
};

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

// The weight fragments of one column tile, K chunk number i in the direction's order.
// (MATS matrices from `first` on)
template <bool TR, int MATS>
__device__ __forceinline__ void rows_weights(const RingTeamArgs& c, int first, int out, int q, bf16x8 (&wt)[MATS][ROWS_CHUNKS]) {
  auto load = [&](auto how) {
    constexpr int HOW = decltype(how)::value, BATCH = HOW == WEIGHT_ROWS4 ? 8 : 4;
#pragma unroll
    for (int mm = 0; mm < MATS; ++mm)
#pragma unroll
      for (int i0 = 0; i0 < ROWS_CHUNKS; i0 += BATCH) {
        WeightLoad l[BATCH];
        const int m = first + mm;
        const float* W = m == 0 ? c.Wo : c.Wa + (size_t)(m - 1) * c.N * c.N;
#pragma unroll
        for (int i = 0; i < BATCH; ++i) weight_load<HOW>(l[i], W, c.N, out, 32 * (TR ? i0 + i : rows_chunk(i0 + i)) + 8 * q);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          bf16x8 f = weight_fragment(l[i], c.N, out, 32 * (TR ? i0 + i : rows_chunk(i0 + i)) + 8 * q, m == 0 ? c.scale0 : 1.f, m == 0 ? c.shift0 : 0.f);
          asm volatile("" : "+v"(f));              // (here, not at its first use: twice the registers until then)
          wt[mm][i0 + i] = f;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  if constexpr (TR) load(std::integral_constant<int, WEIGHT_COLUMNS>{});
  else if ((c.N & 3) == 0) load(std::integral_constant<int, WEIGHT_ROWS4>{});
  else load(std::integral_constant<int, WEIGHT_ROWS>{});
}

// A compute wave's place in the exchange: its operand's chunks in the direction's order.  Rows past the batch are not there.
template <bool TR>
__device__ __forceinline__ void rows_places(const RingTeamArgs& c, int lane, int rows, unsigned (&at)[ROWS_CHUNKS]) {
#pragma unroll
  for (int i = 0; i < ROWS_CHUNKS; ++i) {
    const int kc = TR ? i : rows_chunk(i);
    at[i] = kc < c.KC && (lane & 15) < rows ? (unsigned)kc * CHUNK_BYTES + lane * 16 : NOWHERE;        // (past the contraction: zeros)
  }
}

// Waits until the operand under `base` is complete.
__device__ __forceinline__ void rows_wait(RowsOperand& op, const RingTeamArgs& c, __amdgpu_buffer_rsrc_t rsrc, const unsigned (&at)[ROWS_CHUNKS],
                                          unsigned base, bool& dead, int lane) {
  int spins = 0;
  while (!dead && !op.ready()) {
    if (++spins > c.spin_max) {
      dead = true;
      if (lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
    }
    op.issue(rsrc, at, base);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0), for the compiler's books: this operand has landed on every path
}

// Where an auxiliary thread's two neurons go in the weight-resident kernels' record (split tile order: neuron j is in tile
// 4 (j / 64) + j % 4, column j % 64 / 4), byte offsets inside a batch tile.  After the quad exchange a lane has all four
// rows of neuron j0 + (lane & 1).
struct RowsRecord {
  unsigned d_off, p_off;
  bool row_ok;
  template <int TILES>
  __device__ __forceinline__ RowsRecord(const TeamAux<TILES>& aux, int rows) {
    const int lane = aux.lane, j = aux.j0 + (lane & 1), rq = aux.map.b >> 2, w = j >> 6, n = (j & 63) >> 2, cc = j & 3;
    d_off = (lane & 2) || !aux.map.active ? NOWHERE : (unsigned)((w * 64 + rq * 16 + n) * 32 + cc * 8);
    p_off = aux.map.active ? (unsigned)(((w * 4 + cc) * 64 + rq * 16 + n) * 16 + (lane & 2) * 4) : NOWHERE;
    row_ok = aux.map.active && aux.map.b < rows;
  }
  __device__ __forceinline__ void dact_store(_Float16* base, int t, int nbt, int bt, int lane, unsigned d) const {
    const u32x2 x = quad_rows2(d, lane);
    __builtin_amdgcn_raw_buffer_store_b64(x, team_buffer(base + ((size_t)t * nbt + bt) * 4096, 8192), (int)d_off, 0, 0);
  }
  // steps t (even; otherwise nothing is stored) and t + 1
  __device__ __forceinline__ void pair_store(__bf16* base, int t, bool even, int nbt, int bt, int lane, unsigned lo, unsigned hi) const {
    const u32x2 a = quad_rows2(lo, lane), d = quad_rows2(hi, lane);
    __builtin_amdgcn_raw_buffer_store_b64((lane & 2) ? d : a, team_buffer(base + ((size_t)(t >> 1) * nbt + bt) * 8192, even ? 16384 : 0), (int)p_off, 0, 0);
  }
};

// The two gates of an auxiliary thread's row, where its matrices' sums come apart.  They are read before the barrier that ends the step's
// products, as the compute waves with two tiles do: behind it the first auxiliary wave may already be putting the gates of two steps on
// into the same buffer.
template <int TILES>
__device__ __forceinline__ f32x2 rows_gates(const TeamAux<TILES>& aux, const float* gates) {
  if constexpr (TILES == 1) return f32x2{gates[aux.map.b], gates[16 + aux.map.b]};
  return f32x2{0.f, 0.f};
}

// An auxiliary thread's two sums: of the one share, or of the matrices' with its row's gates.
template <int TILES>
__device__ __forceinline__ void rows_sums(const TeamAux<TILES>& aux, const float* share, f32x2 g, int buf, float (&x)[2]) {
  if constexpr (TILES == 1) {
    using AM = AuxMap<1>;
    const float* src = share + (size_t)buf * ROWS_MATS * AM::SHARE + aux.map.q * AM::QS + aux.map.b * 4 + 2 * aux.map.p;
    f32x2 P[ROWS_MATS];
#pragma unroll
    for (int m = 0; m < ROWS_MATS; ++m) P[m] = *reinterpret_cast<const f32x2*>(src + m * AM::SHARE);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = fmaf(g[1], P[2][i], fmaf(g[0], P[1][i], P[0][i]));
  } else {
    aux.template sum_shares<1>(share, buf, x);
  }
}

template <int ACT, bool SAVE, int TILES>
__device__ __forceinline__ void rows_forward(const RingFwdArgs& p, const RingTeamArgs& c, char* lds) {
  using TA = TeamAux<TILES>;
  using RS = RowsSplit<TILES>;
  using AM = typename TA::AM;
  constexpr int NPT = TA::NPT;
  int team, mem;
  if (!team_coords(c, team, mem)) return;
  const LdsPlan L = lds_plan<TILES, RS::SHARES>(c.k, 1, 0, c.KC, 0, false, false);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const unsigned tile_bytes = (unsigned)c.KC * CHUNK_BYTES, slot_bytes = tile_bytes * (unsigned)c.nbt;
  const unsigned tile_at = (unsigned)team * tile_bytes;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  const int T = p.T, rows = p.B - 16 * team;

  if (w < RS::WAVES) {
    const int q = lane >> 4, b = lane & 15;
    unsigned at[ROWS_CHUNKS];
    rows_places<false>(c, lane, rows, at);
    constexpr int MATS = ROWS_MATS / RS::SHARES;
    bf16x8 wt[MATS][ROWS_CHUNKS];
    rows_weights<false>(c, TILES == 1 ? w : 0, 16 * (mem * TILES + (TILES == 1 ? 0 : w)) + b, q, wt);
    lds_barrier();                                        // the first gates are in LDS
    if (!team_go(lds, L)) return;
    float* const dst = share + w * AM::SHARE + q * AM::QS + b * 4;
    RowsOperand op;
    int slot = 0;
    bool dead = c.spin_max < 0;
    if (dead && lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
    op.issue(rsrc, at, tile_at);
    for (int t = 0; t < T; ++t) {
      const float* g = gl + (t & 1) * c.k * 16 + b;        // (two tiles; with one the auxiliary waves apply the gates)
      const float g1 = TILES == 2 ? g[0] : 0.f, g2 = TILES == 2 ? g[16] : 0.f;
      rows_wait(op, c, rsrc, at, (unsigned)slot * slot_bytes + tile_at, dead, lane);
      f32x4 P0 = {0.f, 0.f, 0.f, 0.f}, P1 = P0, P2 = P0, v;
#pragma unroll
      for (int i = 0; i < ROWS_CHUNKS; ++i) {
        const bf16x8 x = __builtin_bit_cast(bf16x8, op.x[i]);
        if constexpr (TILES == 2) {
          P1 = mfma16(wt[1][i], x, P1);
          P2 = mfma16(wt[2][i], x, P2);
        }
        P0 = mfma16(wt[0][i], x, P0);
      }
      if constexpr (TILES == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaf(g2, P2[i], fmaf(g1, P1[i], P0[i]));
      } else {
        v = P0;
      }
      *reinterpret_cast<f32x4*>(dst + (t & 1) * (RS::WAVES * AM::SHARE)) = v;
      slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
      lds_barrier();
      team_look(c.look);
      op.issue(rsrc, at, (unsigned)slot * slot_bytes + tile_at);      // (the first look at the next state)
    }
    return;
  }

  __builtin_amdgcn_s_setprio(3);
  TA aux(c, mem, tid - 64 * RS::WAVES);
  team_arrive(c, team, aux.at);
  const RowsRecord rec(aux, rows);
  const int N = p.N, B = p.B;
  const float oma = 1.f - p.alpha;
  const ActScale asc = act_scale_make(p.alpha);
  const unsigned d_mask = rec.row_ok ? (aux.j0 < N ? 0xFFFFu : 0u) | (aux.j0 + 1 < N ? 0xFFFF0000u : 0u) : 0u;
  const bool late_once = c.rows == 2 && (aux.j0 & 32);
  const unsigned x_off = rec.row_ok ? aux.x_off : NOWHERE;
  auto put = [&](int slot, unsigned x) { __builtin_amdgcn_raw_buffer_store_b32(x, rsrc, (int)x_off, (int)((unsigned)slot * slot_bytes + tile_at), ST_LOCAL); };
  float r[NPT];
  aux.row_load(p.r_init, N, B, team, r);
  unsigned before = pack_bf16(r[0], r[1]);
  put(0, not_empty(before));
  const TeamGates tg(c, aux.at);
  auto gates_of = [&](int t) { return tg.fetch(c, t < T ? t : T - 1, team); };
  tg.put(gl, gates_of(0));
  float gA = gates_of(1), gB = gates_of(2);
  team_gather(c, lds, L, team, aux.at);
  lds_barrier();
  if (!team_go(lds, L)) return;

  int slot = 0, t = 0;
  auto step = [&](bool even, float& g) {
    const f32x2 row_gates = rows_gates<TILES>(aux, gl + (t & 1) * c.k * 16);
    tg.put(gl + ((t + 1) & 1) * c.k * 16, g);               // the next step's gates, fetched two steps ago
    lds_barrier();                                          // the step's products are complete
    float x[NPT], rn[NPT], aF[NPT];
    rows_sums<TILES>(aux, share, row_gates, t & 1, x);
    ActRecord<ACT> rd[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) aF[i] = rd[i].apply(x[i], asc);
#pragma unroll
    for (int i = 0; i < NPT; ++i) rn[i] = aux.j0 + i < N ? fmaf(oma, r[i], aF[i]) : 0.f;
    const int next_slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
    const unsigned now = pack_bf16(rn[0], rn[1]);
    put(next_slot, not_empty(now));                         // (after the last step: nobody looks)
    g = gates_of(t + 3);
    put(slot == 0 ? ROWS_SLOTS - 1 : slot - 1, EMPTY);
    aux.row_store(p.hist + (size_t)t * B * N, N, B, team, rn);
    if constexpr (SAVE) {
      rec.dact_store(p.dfrag, t, p.nbt, team, lane, ActRecord<ACT>::pair(asc, rd[0], rd[1], late_once && t + 1 < T) & d_mask);
      if (even) rec.pair_store(p.rfrag, t, true, p.nbt, team, lane, before, t + 1 < T ? now : 0u);
      before = now;
    }
#pragma unroll
    for (int i = 0; i < NPT; ++i) r[i] = rn[i];
    slot = next_slot;
    ++t;
  };
  while (t < T) {
    step(true, gA);
    if (t >= T) return;
    step(false, gB);
  }
}

}  // namespace

template <int ACT, int TILES>
__global__ __launch_bounds__(64 * (RowsSplit<TILES>::WAVES + AUX)) __attribute__((amdgpu_waves_per_eu(2, 2))) void ring_team_rows_kernel(RingFwdArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  rows_forward<ACT, false, TILES>(p, c, lds);
}

// With the weight-resident kernels' record.
template <int ACT, int TILES>
__global__ __launch_bounds__(64 * (RowsSplit<TILES>::WAVES + AUX)) __attribute__((amdgpu_waves_per_eu(2, 2))) void ring_team_res256_fwd_kernel(RingFwdArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  rows_forward<ACT, true, TILES>(p, c, lds);
}

// ------------------------------------------------------------------------------------------------
// BPTT.  Operand number s is g of step T - 1 - s, the products of round s give the carry into step T - 2 - s.  The ungated
// sum starts from (1 - alpha) G: the auxiliary waves leave it in LDS before they publish g, so a wave that has seen all of g
// finds it there.
// ------------------------------------------------------------------------------------------------
template <bool GA, int TILES>
__global__ __launch_bounds__(64 * (RowsSplit<TILES>::WAVES + AUX)) __attribute__((amdgpu_waves_per_eu(2, 2))) void ring_team_res256_bptt_kernel(RingBpttArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  using TA = TeamAux<TILES>;
  using RS = RowsSplit<TILES>;
  using AM = typename TA::AM;
  constexpr int NPT = TA::NPT;
  int team, mem;
  if (!team_coords(c, team, mem)) return;
  const LdsPlan L = lds_plan<TILES, RS::SHARES>(c.k, 1, 0, c.KC, 0, true, GA);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const unsigned tile_bytes = (unsigned)c.KC * CHUNK_BYTES, slot_bytes = tile_bytes * (unsigned)c.nbt;
  const unsigned tile_at = (unsigned)team * tile_bytes;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const keep = reinterpret_cast<float*>(lds + L.state);        // (1 - alpha) G: [tile][q][row] x 4 neurons
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  float* const prev = reinterpret_cast<float*>(lds + L.rows);         // r_prev of a round's step, two buffers, likewise
  float* const ga = reinterpret_cast<float*>(lds + L.ga);             // dL/dA shares [2][channel][tile][row]
  const int T = p.T, rows = p.B - 16 * team;
  const int steps = (p.grad_r_init || GA) ? T : T - 1;

  if (w < RS::WAVES) {
    const int q = lane >> 4, b = lane & 15;
    unsigned at[ROWS_CHUNKS];
    rows_places<true>(c, lane, rows, at);
    constexpr int MATS = ROWS_MATS / RS::SHARES;
    const int tile = TILES == 1 ? 0 : w;
    bf16x8 wt[MATS][ROWS_CHUNKS];
    rows_weights<true>(c, TILES == 1 ? w : 0, 16 * (mem * TILES + tile) + b, q, wt);
    lds_barrier();                                        // the first gates (and r_prev) are in LDS
    if (!team_go(lds, L)) return;
    float* const dst = share + w * AM::SHARE + q * AM::QS + b * 4;
    RowsOperand op;
    int slot = 0;
    bool dead = c.spin_max < 0;
    if (dead && lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
    op.issue(rsrc, at, tile_at);
    for (int s = 0; s < steps; ++s) {
      const float* g = gl + (s & 1) * c.k * 16 + b;
      const float g1 = TILES == 2 ? g[0] : 0.f, g2 = TILES == 2 ? g[16] : 0.f;
      rows_wait(op, c, rsrc, at, (unsigned)slot * slot_bytes + tile_at, dead, lane);
      asm volatile("" ::: "memory");                       // (what follows is read behind the wait)
      f32x4 P0 = *reinterpret_cast<const f32x4*>(keep + (tile * 64 + lane) * 4);
      f32x4 P1 = {0.f, 0.f, 0.f, 0.f}, P2 = P1, v;
      if (TILES == 1 && w > 0) P0 = P1;                    // (this wave's matrix is a gated one)
      if constexpr (TILES == 2) {
#pragma unroll
        for (int i = 0; i < ROWS_CHUNKS; ++i) {
          const bf16x8 x = __builtin_bit_cast(bf16x8, op.x[i]);
          P1 = mfma16(wt[1][i], x, P1);
          P2 = mfma16(wt[2][i], x, P2);
        }
      }
#pragma unroll
      for (int i = 0; i < ROWS_CHUNKS; ++i) P0 = mfma16(wt[0][i], __builtin_bit_cast(bf16x8, op.x[i]), P0);
      if constexpr (TILES == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaf(g2, P2[i], fmaf(g1, P1[i], P0[i]));
      } else {
        v = P0;
      }
      *reinterpret_cast<f32x4*>(dst + (s & 1) * (RS::WAVES * AM::SHARE)) = v;
      if constexpr (GA) {
        const f32x4 rp = *reinterpret_cast<const f32x4*>(prev + ((s & 1) * TILES * 64 + tile * 64 + lane) * 4);
        float* const gp = ga + ((s & 1) * 2 * TILES + tile) * 16 + b;
        auto dot = [&](const f32x4& P, int ch) {
          float d = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) d = fmaf(P[i], rp[i], d);
          d = sum_bits45(d);
          if (lane < 16) gp[ch * TILES * 16] = d;
        };
        if constexpr (TILES == 2) {
          dot(P1, 0);
          dot(P2, 1);
        } else if (w > 0) {
          dot(P0, w - 1);
        }
      }
      lds_barrier();
      slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
      team_look(c.look);
      op.issue(rsrc, at, (unsigned)slot * slot_bytes + tile_at);      // (the first look at the next one)
    }
    return;
  }

  __builtin_amdgcn_s_setprio(3);
  TA aux(c, mem, tid - 64 * RS::WAVES);
  team_arrive(c, team, aux.at);
  const RowsRecord rec(aux, rows);
  const int N = p.N, B = p.B, nbt = p.nbt;
  const float oma = 1.f - p.alpha;
  const bool loss = p.loss_coef != nullptr;
  const unsigned x_off = rec.row_ok ? aux.x_off : NOWHERE;
  auto put = [&](int slot, unsigned x) { __builtin_amdgcn_raw_buffer_store_b32(x, rsrc, (int)x_off, (int)((unsigned)slot * slot_bytes + tile_at), ST_LOCAL); };
  const TeamGates tg(c, aux.at);
  float cs[NPT] = {0.f, 0.f}, sn[NPT] = {0.f, 0.f}, up = 0.f;
  if (loss) {
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const float phi = 6.2831853071795864769f * (float)(aux.j0 + i) / (float)N;
      cs[i] = cosf(phi);
      sn[i] = sinf(phi);
    }
    up = (p.loss_upstream ? p.loss_upstream[0] : 1.f) * p.loss_inv_rows;
  }
  const float* const grads = loss ? p.hist : p.grad_out;
  const int at_row = 16 * team + (rec.row_ok ? aux.map.b : rows - 1);
  const char* const coef = loss ? reinterpret_cast<const char*>(p.loss_coef + at_row) : reinterpret_cast<const char*>(c.Wo);
  const int j = aux.j0, dw = j >> 6, dn = (j & 63) >> 2;
  const unsigned d_at = (unsigned)((dw * 64 + (aux.map.b >> 2) * 16 + dn) * 16 + (j & 3) * 4 + (aux.map.b & 3));     // fp16 values
  const int at4 = (aux.map.c * 64 + aux.map.q * 16 + aux.map.b) * 4 + 2 * aux.map.p;        // of the thread's values in keep and prev
  struct In {                          // of a step: grad_output or history, record, loss coefficients, r_prev, gate
    float go[NPT];
    _Float16 d[NPT];
    f32x3 cf;
    float rp[GA ? NPT : 1];
    float g;
  };
  auto fetch = [&](int t, In& in) {
    const int tc = t < 0 ? 0 : t;
    aux.row_load_raw(grads + (size_t)tc * B * N, N, B, team, in.go);
    const _Float16* src = p.dfrag + ((size_t)tc * nbt + team) * 4096 + d_at;
    in.d[0] = src[0];
    in.d[1] = src[4];
    in.cf = *reinterpret_cast<const f32x3*>(coef + (loss ? (size_t)tc * B * 16 : 0));      // (without the loss head: unused)
    in.g = tg.fetch(c, tc, team);
    if constexpr (GA) aux.row_load_raw(tc == 0 ? p.r_init : p.hist + (size_t)(tc - 1) * B * N, N, B, team, in.rp);
  };
  auto put_side = [&](int buf, const In& in) {
    tg.put(gl + buf * c.k * 16, in.g);
    if constexpr (GA) {
      float v[NPT] = {in.rp[0], in.rp[1]};
      aux.align(N, v);
#pragma unroll
      for (int i = 0; i < NPT; ++i) if (aux.map.active) prev[buf * TILES * 256 + at4 + i] = rec.row_ok && j + i < N ? (float)(__bf16)v[i] : 0.f;
    }
  };
  const bool ok[NPT] = {rec.row_ok && j < N, rec.row_ok && j + 1 < N};
  // what is carried into the step -> g's bf16 pair; (1 - alpha) G into LDS, where it is before this returns
  auto form_g = [&](const In& in, const float (&carry)[NPT]) {
    float gin[NPT] = {in.go[0], in.go[1]};
    aux.align(N, gin);
    const float kc = in.cf[0] * up, ks = in.cf[1] * up, beta = in.cf[2] * up;
    float gg[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const float r = gin[i], of_loss = fmaf(kc, cs[i], fmaf(ks, sn[i], r > 0.f ? beta : (r < 0.f ? -beta : 0.f)));
      const float all = (loss ? of_loss : r) + carry[i];
      const float G = ok[i] ? all : 0.f, g = (float)in.d[i] * G;
      if (aux.map.active) keep[at4 + i] = oma * G;
      gg[i] = ok[i] ? g : 0.f;                    // the record carries alpha
    }
    const unsigned x = pack_bf16(gg[0], gg[1]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    return x;
  };
  // dL/dA of round s: one partial per column tile
  auto flush = [&](int s) {
    if constexpr (GA) {
      const int at = aux.at, tile = TILES == 1 ? 0 : at >> 5 & 1, ch = at >> 4 & 1, row = at & 15, t = T - 1 - s;
      const float v = ga[((s & 1) * 2 * TILES + (ch * TILES + tile)) * 16 + row];
      const __amdgpu_buffer_rsrc_t r = team_buffer(c.ga_part + ((size_t)mem * TILES * T + t) * 2 * B, ((size_t)T + 1) * 2 * B * 4);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r,
                                            (int)(at < 32 * TILES && row < rows ? (unsigned)((tile * T * 2 + ch) * B + 16 * team + row) * 4 : NOWHERE), 0, 0);
    }
  };

  In inA, inB;
  fetch(T - 1, inA);
  fetch(T - 2, inB);
  put_side(0, inA);
  unsigned x;
  {
    const float zero[NPT] = {0.f, 0.f};
    x = form_g(inA, zero);
    put(0, not_empty(x));
  }
  unsigned held = 0;
  rec.pair_store(p.gfrag, T - 1, (T & 1) != 0, nbt, team, lane, x, 0u);
  held = x;                            // (read at even steps: the odd one's behind them)
  fetch(T - 3, inA);
  team_gather(c, lds, L, team, aux.at);
  lds_barrier();
  if (steps == 0 || !team_go(lds, L)) return;

  const __amdgpu_buffer_rsrc_t rinit = team_buffer(p.grad_r_init + (size_t)16 * team * N, p.grad_r_init ? (size_t)(rows < 16 ? rows : 16) * N * 4 : 0);
  int slot = 0, s = 0;
  auto round = [&](In& in) {
    const f32x2 row_gates = rows_gates<TILES>(aux, gl + (s & 1) * c.k * 16);
    put_side((s + 1) & 1, in);                               // the gates (and r_prev) of the next round, which is this set's step's
    lds_barrier();                                          // the round's products are complete
    float carry[NPT];
    rows_sums<TILES>(aux, share, row_gates, s & 1, carry);
#pragma unroll
    for (int i = 0; i < NPT; ++i) carry[i] = ok[i] ? carry[i] : 0.f;
    const int t = T - 2 - s, tt = t < 0 ? 0 : t, next_slot = slot + 1 == ROWS_SLOTS ? 0 : slot + 1;
    // (no branches: what a round has nothing to store for is dropped, so that a wait for a load counts what is behind it)
    x = form_g(in, carry);
    put(next_slot, not_empty(x));                            // (after the last round: nobody looks)
    fetch(t - 2, in);
    put(slot == 0 ? ROWS_SLOTS - 1 : slot - 1, EMPTY);
    rec.pair_store(p.gfrag, tt, t >= 0 && (t & 1) == 0, nbt, team, lane, x, t + 1 < T ? held : 0u);
    held = x;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, carry[0]), rinit, (int)(t < 0 ? aux.row_off : NOWHERE), 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, carry[1]), rinit, (int)(t < 0 && j + 1 < N ? aux.row_off + 4 : NOWHERE), 0, 0);
    flush(s);
    slot = next_slot;
    ++s;
  };
  while (s < steps) {
    round(inB);
    if (s >= steps) return;
    round(inA);
  }
}

// Sum of the column tiles' dL/dA partials: the sixteen lanes of a row group, the four waves.
__global__ __launch_bounds__(256) void ring_team_res256_ga_reduce_kernel(const float* __restrict__ part, float* __restrict__ grad_A, int T, int B) {
  const size_t n = (size_t)T * 2 * B, u = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= n) return;
  float v[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float* src = part + (size_t)4 * w * n + u;
    v[w] = (src[0] + src[n]) + (src[2 * n] + src[3 * n]);
  }
  const int b = (int)(u % B);
  const size_t tc = u / B;
  grad_A[((size_t)b * T + (tc >> 1)) * 2 + (tc & 1)] = ((v[0] + v[1]) + v[2]) + v[3];
}

// record: with one, or a BPTT; then all 256 neurons have a member (the padding's part of the record is zero)
RingTeamPlan ring_team_rows_plan(int N, int k, int B, bool record, int launches) {
  RingTeamPlan p{};
  if (!ring_res256_applicable(N, k)) return p;
  p.KC = record ? ROWS_CHUNKS : (N + 31) / 32;
  p.nteams = (B + 15) / 16;
  const int one = 2 * p.KC, tiles = p.nteams <= 8 * (32 / (launches * one)) ? 1 : 2;
  p.G = (one + tiles - 1) / tiles;
  p.nt = 1;
  p.slots = ROWS_SLOTS;
  p.ok = p.nteams <= 8 * (32 / p.G);                       // (8 XCDs of 32 compute units)
  p.shape = RingTeamShape{ROWS_CHUNKS, tiles, ROWS_MATS, tiles == 1 ? RowsSplit<1>::WAVES : RowsSplit<2>::WAVES, 0, 8 * p.G * ((p.nteams + 7) / 8)};
  p.xchg_bytes = (size_t)ROWS_SLOTS * p.nteams * p.KC * CHUNK_BYTES;
  p.gather_bytes = (size_t)p.nteams * RING_TEAM_WORD * sizeof(unsigned long long);
  return p;
}

size_t ring_team_rows_ga_bytes(int T, int B) { return (size_t)16 * T * 2 * B * sizeof(float); }

template <int TILES, typename Args, typename Kernel>
static hipError_t rows_start(Kernel kern, const Args& a, const RingTeamArgs& c, const RingTeamShape& sh, bool bptt, bool ga, hipStream_t st) {
  const unsigned lds = lds_plan<TILES, RowsSplit<TILES>::SHARES>(c.k, 1, 0, c.KC, 0, bptt, ga).total + (ga ? RowsSplit<TILES>::GA_MORE : 0);
  return ring_team_start(reinterpret_cast<const void*>(kern), sh, c.G, lds, st,
                         [&](dim3 g, dim3 b, unsigned bytes) { RING_LAUNCH(kern, g, b, bytes, st, a, c); });
}

template <int TILES>
static hipError_t launch_rows(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  auto go = [&](auto kern) { return rows_start<TILES>(kern, a, c, sh, false, false, st); };
  switch (a.act) {
    case ACT_RELU: return a.dfrag ? go(ring_team_res256_fwd_kernel<ACT_RELU, TILES>) : go(ring_team_rows_kernel<ACT_RELU, TILES>);
    case ACT_GELU: return a.dfrag ? go(ring_team_res256_fwd_kernel<ACT_GELU, TILES>) : go(ring_team_rows_kernel<ACT_GELU, TILES>);
    case ACT_TANH: return a.dfrag ? go(ring_team_res256_fwd_kernel<ACT_TANH, TILES>) : go(ring_team_rows_kernel<ACT_TANH, TILES>);
    case ACT_SILU: return a.dfrag ? go(ring_team_res256_fwd_kernel<ACT_SILU, TILES>) : go(ring_team_rows_kernel<ACT_SILU, TILES>);
    default: return hipErrorInvalidValue;
  }
}

hipError_t ring_launch_team_rows(const RingFwdArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  return sh.c16 == 1 ? launch_rows<1>(a, c, sh, st) : launch_rows<2>(a, c, sh, st);
}

hipError_t ring_launch_team_rows_bptt(const RingBpttArgs& a, const RingTeamArgs& c, const RingTeamShape& sh, hipStream_t st) {
  const bool ga = a.grad_A != nullptr;
  if (sh.c16 == 1)
    return ga ? rows_start<1>(ring_team_res256_bptt_kernel<true, 1>, a, c, sh, true, true, st)
              : rows_start<1>(ring_team_res256_bptt_kernel<false, 1>, a, c, sh, true, false, st);
  return ga ? rows_start<2>(ring_team_res256_bptt_kernel<true, 2>, a, c, sh, true, true, st)
            : rows_start<2>(ring_team_res256_bptt_kernel<false, 2>, a, c, sh, true, false, st);
}

hipError_t ring_launch_team_rows_ga(const float* part, float* grad_A, int T, int B, hipStream_t st) {
  const size_t n = (size_t)T * 2 * B;
  hipLaunchKernelGGL(ring_team_res256_ga_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, part, grad_A, T, B);
  return hipGetLastError();
}
