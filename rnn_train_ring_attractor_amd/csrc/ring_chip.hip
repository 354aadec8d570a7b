// Chip kernels: the forward without a saved record for wide rings (512 < N <= 2048), the weights kept in the registers and LDS
// of ALL compute units for the whole sequence, the state handed over between the XCDs once per step.
//
// What bounds the step-per-launch kernels here (ring_panel.hip) is that every step pulls all (1 + a_dim) N^2 weights from
// beyond L2 again and waits for a launch: at N = 2048 with 12 channels 109 MB a step.  The chip holds 128 MB of registers and
// 40 MB of LDS.  Beside what a step works with there is room for 16 channels up to N = 1536 and for 13 up to N = 2048 (117 MB).  A
// member (a workgroup) keeps all matrices of NPW = 8, 16 or 32 neurons; G = N / NPW members make a row group, which takes every
// nrg-th batch tile of 16 rows through the sequence.  Fewer neurons per member spread the weights over more compute units, more let
// several row groups work side by side, each reading the state of its own rows only.
//
//   * Eight waves split the contraction as in ring_team.hpp (wave w owns K chunks w, w + 8, ...); a wave loads just its chunks of the
//     state, multiplies them with its resident fragments (weights are the A operand: a lane ends up with four neurons of one batch
//     row), gates and sums over the matrices in fp32 and leaves one share per neuron in LDS.
//   * With eight neurons a column tile of 16 holds two matrices side by side, else one.  Either way the even and the odd matrices
//     are summed apart and added up last, so that a row's bits depend on N and a_dim only, not on the batch it is in.
//   * Behind the item's barrier every wave adds the shares of its two rows in wave order, applies the activation, publishes the new
//     state and writes the history.  There is no auxiliary wave as in ring_team.hpp: all registers hold weights.  One wave per
//     item in turn, whose stores held up its next operand (one in-order counter): N = 1100, 2 channels, B = 1 3.9 against 3.2 us
//     per step, N = 700, 6 channels, B = 1 3.4 against 3.0.  All waves issue the same operations, so the compiler waits for
//     an operand's loads and not for the stores behind them.
// What bounds an item (step, tile of 16 rows) with several tiles per group is instructions.  Cycles of a wave's item at N = 1024, 6
// channels, B = 256 (N = 640 to 1100, B = 512 and 1024: 2900 to 3800): 3250, of them products with the gates 1500, epilogue 890, barrier 550,
// waiting for the state 300; a compute unit takes in 13 bytes a cycle.  With one tile it is the hand-over: 6600 to 8400 of 9200 to
// 11300 cycles (N = 640 to 2048) are the epilogue, which publishes and then waits to poll, and the wait for the state.
//
// Exchange: the protocol of ring_team.hpp (the data is its own flag, slots refilled with a pattern no state can be), but with
// stores that go through to where all XCDs see them.  Measured for 256 members and one tile: 1.9 us from step to step, 2.6 with
// one reader per XCD that hands on inside it, 5.0 with flags beside the data.  Polling competes with the stores it waits for:
// a barrier before the first poll and a pause between polls took N = 2048, 2 channels, B = 16 from 9.7 to 5.9 us per step.
// A refill is in place before its slot is polled again.  A wave stores the same rows of a tile for the whole sequence.  It issues
// a refill in the epilogue of item i; the operand of item i + DEPTH (the first that it asks for behind that) it waits for before
// that item's epilogue, and memory operations complete in order: what it publishes from there on is published behind the refill.
// A reader polls for state s - 1 + slots only after state s - 2 + slots of the same rows, published (slots - 3) rounds of the
// group's tiles after item i, which is at least DEPTH items: 5 with one tile and 8 slots, 3 with two (one in the smaller groups)
// and 6, 6 with three (two) and 6, 3 from four (three) up and 4.
//
// Residence: as in ring_team.hpp a row group counts itself before the time loop and gives up as a whole if it is not complete in
// time; ring_chip_rest_kernel behind this launch does the tiles of groups that gave up, with the same bits, on what compute units
// there are.
#include "ring_team.hpp"

#include <stdlib.h>
#include <algorithm>

namespace {

constexpr int ST_THROUGH = 16;        // sc1: visible to the other XCDs
constexpr size_t CHIP_LDS = 160 * 1024;
constexpr unsigned long long CHIP_GAVE_UP = 1ull << 63;
constexpr int W = 8;                  // waves
constexpr int CHIP_QS = 72;           // LDS floats between the neuron quads of a share (bank spread)

struct RingChipArgs {
  const float *A, *Wo, *Wa, *r_init;
  float* hist;
  void* xchg;                    // [slots][batch tiles][K chunks][1280 bytes], all 0xFF at launch
  // A word per row group, 0 at launch: members that are resident; top bit: given up.  Behind them ring_chip_rest_kernel's, 0 at launch:
  // units drawn, and per tile block those that are done.
  unsigned long long* gather;
  int* host_err;
  unsigned xchg_bytes;
  float J0, J1, alpha;
  int N, k, T, B, nbt, KC, G, nrg, nt, slots, act, spin_max, gather_ticks;
};

// Fragments of a wave: F, of which FR in registers and the rest in LDS, spread evenly over a column tile's products.
// DEPTH: operands on their way or in use.  1: the next item's is asked for behind this one's epilogue (one tile per group or two: it
// cannot be there earlier); 2 and 3: before its products, one item or two ahead (see chip_plan).
template <int NPW, int KPW, int CT, int DEPTH>
struct ChipShape {
  static constexpr int F = CT * KPW;
  static constexpr int ROOM = (256 - 44 - DEPTH * 5 * KPW) / 4;
  static constexpr int FR = F <= ROOM ? F : ROOM - 4;           // (parked ones cost registers on their way)
  static constexpr int P = F - FR;                              // parked in LDS
  // column tiles without a gap in all calls that take this number of them (see RING_CHIP_SHAPES: the smallest that is enough)
  static constexpr int FULL = NPW == 8 ? (CT == 2 ? 1 : CT == 4 ? 2 : CT == 7 ? 4 : 7) : NPW == 16 ? (CT == 3 ? 2 : CT == 4 ? 4 : 5) : (CT == 6 ? 4 : 8);
  static constexpr int SHARE = NPW / 4 * CHIP_QS;               // floats of one wave's share
  static constexpr int MATS = NPW == 8 ? 2 * CT : (NPW == 16 ? CT : CT / 2);      // matrices that there is room for
  static constexpr int LEAST = NPW == 8 ? 2 * FULL : (NPW == 16 ? FULL : FULL / 2);      // and that fill the tiles without a gap
  // Up to three channels at N <= 1024 the teams take every call with few tiles per row group: fewer than three with 32 neurons a member
  // and three channels, fewer than five else.
  static constexpr int TEAMS_UP_TO = KPW > 4 || MATS > 4 ? 0 : (NPW == 32 && KPW == 4 && CT == 8 ? 2 : 4);
  static constexpr bool BUILT = DEPTH == 1 ? TEAMS_UP_TO < 2 : DEPTH == 2 ? P * W <= 144 && TEAMS_UP_TO < 4 : P == 0;
  static constexpr int before(int f) { return f * P / F; }                        // parked ones among the first f
  static constexpr bool is_parked(int f) { return before(f + 1) > before(f); }
};

struct ChipLds { unsigned share, gates, state, go, parked, total; };

__host__ __device__ inline ChipLds chip_lds(int npw, int mats, int parked, int nt) {
  ChipLds p;
  unsigned at = 0;
  p.share = at;
  at += 2u * W * (npw / 4) * CHIP_QS * 4;
  p.gates = at;
  at += 2u * mats * 16 * 4 + 64;                          // (and the spare words of idle threads)
  p.state = at;
  at += (unsigned)nt * W * 64 * 4;
  p.go = at;
  at += 64;
  p.parked = at;
  at += (unsigned)parked * W * 1024;
  p.total = at;
  return p;
}

__device__ __forceinline__ float chip_act(int act, float x) {
  float F, D;
  switch (act) {
    case ACT_RELU: act_fast<ACT_RELU>(x, F, D); break;
    case ACT_GELU: act_fast<ACT_GELU>(x, F, D); break;
    case ACT_TANH: act_fast<ACT_TANH>(x, F, D); break;
    default: act_fast<ACT_SILU>(x, F, D); break;
  }
  return F;
}

// Sum with the lane that differs in lane bit 5.
__device__ __forceinline__ float sum_bit5(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const unsigned a0 = a[0], a1 = a[1];
  return __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
}

// Four neurons' sum as the row sums of eight are made of.
__device__ __forceinline__ float sum4(const f32x4& v) { return (v[0] + v[1]) + (v[2] + v[3]); }

// Four consecutive floats of a row of N, 4-byte aligned; past the end: zero.  Reads stay inside the row.
__device__ __forceinline__ f32x4 row_quad(const float* row, int N, int j) {
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = row[j + i < N ? j + i : N - 1];
    v[i] = j + i < N ? a : 0.f;
  }
  return v;
}

// What a wave multiplies in one item: its K chunks w, w + W, ... of the state and their row sums, asked for together.  The last two
// can lie past the contraction: their lanes then point past the buffer and read zero.
struct ChipOperandAt { unsigned x, rs, x_last[2], rs_last[2]; };
template <int KPW>
struct ChipOperand {
  u32x4 x[KPW];
  unsigned rs[KPW];            // lane (q, row): the row sum over neurons 8q .. 8q + 7 of the chunk
  // (the memory clobber keeps a load from being folded into the same one a poll earlier)
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rsrc, const ChipOperandAt& at, unsigned base) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) {
      const int last = kk - (KPW - 2);
      x[kk] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(last < 0 ? at.x : at.x_last[last < 0 ? 0 : last]), (int)(base + kk * W * CHUNK_BYTES), LD_COHERENT);
      rs[kk] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(last < 0 ? at.rs : at.rs_last[last < 0 ? 0 : last]), (int)(base + kk * W * CHUNK_BYTES), LD_COHERENT);
    }
  }
  __device__ __forceinline__ bool ready() const {
    unsigned m = 0, n = 0;                // (three at a time)
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) {
      m = max(max(m, x[kk][0]), x[kk][1]);
      n = max(max(n, x[kk][2]), x[kk][3]);
      if (kk & 1) m = max(max(m, rs[kk]), rs[kk - 1]);
      else if (kk + 1 == KPW) m = max(m, rs[kk]);
    }
    return __ballot(max(m, n) == EMPTY) == 0;
  }
};

// Where an item's tile lies in something that has `tile` bytes a tile and `step` bytes a step: kept by additions, not multiplied
// out for every item (its scalar arithmetic was a third of the instructions of an item).
struct ChipCursor {
  int j, t;
  const char* at;          // the tile's first byte
  const char* row;         // the step's first tile
  __device__ __forceinline__ void advance(int my_nt, size_t tile, size_t step) {
    const bool wrap = j + 1 == my_nt;
    row = wrap ? row + step : row;
    at = wrap ? row : at + tile;
    j = wrap ? 0 : j + 1;
    t += wrap ? 1 : 0;
  }
};

}  // namespace

template <int NPW, int KPW, int CT, int DEPTH>
__global__ __launch_bounds__(64 * W) void ring_chip_fwd_kernel(RingChipArgs c) {
  using S = ChipShape<NPW, KPW, CT, DEPTH>;
  constexpr int F = S::F, FR = S::FR, P = S::P, RING = P < 3 ? (P ? P : 1) : 3, HALVES = NPW == 32 ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // a row group has 8 / nrg XCDs to itself (workgroups go to XCDs round robin)
  const int per = 8 / c.nrg, x = blockIdx.x & 7, rg = x % c.nrg, mem = (blockIdx.x >> 3) * per + x / c.nrg;
  if (mem >= c.G) return;
  const ChipLds L = chip_lds(NPW, S::MATS, P, c.nt);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4, b = lane & 15;
  const int N = c.N, B = c.B, T = c.T, k = c.k;
  const int my_nt = (c.nbt - rg + c.nrg - 1) / c.nrg;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c.xchg, 0, (int)c.xchg_bytes, 0x00020000);
  const unsigned tile_bytes = (unsigned)c.KC * CHUNK_BYTES, slot_bytes = tile_bytes * (unsigned)c.nbt;
  float* const share = reinterpret_cast<float*>(lds + L.share);
  float* const gl = reinterpret_cast<float*>(lds + L.gates);
  float* const state = reinterpret_cast<float*>(lds + L.state);
  bf16x8* const parked = reinterpret_cast<bf16x8*>(lds + L.parked) + (size_t)w * P * 64 + lane;

  // ---- a lane's output: neuron mem * NPW + on of row orow of a tile (two rows a wave) ----
  const int on = lane % NPW, orow = 2 * w + lane / NPW, oj = mem * NPW + on;
  const bool has_out = lane < 2 * NPW;
  // its place in a tile's exchange area: even neurons store a pair, the second of eight their sum
  const unsigned okc = (unsigned)oj >> 5, o8 = ((unsigned)oj >> 3) & 3;
  const unsigned xoff = !has_out ? NOWHERE
                        : (on & 1) == 0 ? okc * CHUNK_BYTES + (o8 * 16 + orow) * 16 + (oj & 7) * 2
                        : (on & 7) == 1 ? okc * CHUNK_BYTES + 1024 + orow * 16 + o8 * 4 : NOWHERE;
  const unsigned hoff = has_out && oj < N ? (unsigned)(orow * N + oj) * 4 : NOWHERE;
  // what it stores there: the pair as bf16, or the sum in the order (0 + 1) + (2 + 3) + ((4 + 5) + (6 + 7))
  auto published = [&](float v) {
    const float other = __builtin_bit_cast(float, dpp_xor1(__builtin_bit_cast(unsigned, v)));
    float sum = v + other;
    sum += __builtin_bit_cast(float, dpp_xor2(__builtin_bit_cast(unsigned, sum)));
    sum += dpp_ror<0x141>(sum);        // (row_half_mirror: the other four)
    return not_empty((on & 1) == 0 ? pack_bf16(v, other) : __builtin_bit_cast(unsigned, sum));
  };

  // ---- residence, initial state ----
  unsigned long long* const word = c.gather + (size_t)rg * RING_TEAM_WORD;
  if (tid == 0) {
    if (c.gather_ticks < 0) __hip_atomic_fetch_or(word, CHIP_GAVE_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  float* const my_state = state + tid;                       // [tile][thread]
  for (int j = 0; j < my_nt; ++j) {
    const int bt = rg + c.nrg * j, row = 16 * bt + orow;
    const float v = c.r_init[(size_t)(row < B ? row : B - 1) * N + (oj < N ? oj : N - 1)], r = has_out && row < B && oj < N ? v : 0.f;
    my_state[j * 64 * W] = r;
    __builtin_amdgcn_raw_buffer_store_b32(published(r), rsrc, (int)xoff, (int)((unsigned)bt * tile_bytes), ST_THROUGH);
  }

  // ---- weights ----
  bf16x8 wreg[FR];
  auto load_weights = [&](auto how) {
    auto place = [&](int f, int& m, int& out, int& k0) {
      const int ct = f / KPW;
      k0 = 32 * (w + W * (f % KPW)) + 8 * q;
      asm volatile("" : "+v"(k0));         // (or addresses and masks are kept from one column tile to the next: registers)
      if constexpr (NPW == 8) { m = 2 * ct + (b >> 3); out = mem * 8 + (b & 7); }
      else if constexpr (NPW == 16) { m = ct; out = mem * 16 + b; }
      else { m = ct >> 1; out = mem * 32 + 16 * (ct & 1) + b; }
    };
    auto load = [&](WeightLoad& l, int f) {
      int m, out, k0;
      place(f, m, out, k0);
      weight_load<decltype(how)::value>(l, m == 0 || m > k ? c.Wo : c.Wa + (size_t)(m - 1) * N * N, N, out, k0);
    };
    auto keep = [&](const WeightLoad& l, int f) {
      int m, out, k0;
      place(f, m, out, k0);
      bf16x8 v = weight_fragment(l, m <= k ? N : 0, out, k0, 1.f, 0.f);
      asm volatile("" : "+v"(v));          // (converted here, not at its first use)
      const int at = S::before(f);
      if (S::is_parked(f)) parked[at * 64] = v;
      else wreg[S::is_parked(f) ? 0 : f - at] = v;
    };
    constexpr int BATCH = 6;
    WeightLoad l[BATCH];
#pragma unroll
    for (int f = 0; f < BATCH && f < F; ++f) load(l[f], f);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      keep(l[f % BATCH], f);
      if (f + BATCH < F) load(l[f % BATCH], f + BATCH);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if ((N & 3) == 0) load_weights(std::integral_constant<int, WEIGHT_ROWS4>{});
  else load_weights(std::integral_constant<int, WEIGHT_ROWS>{});
  bf16x8 ring[RING];                       // the next parked fragments, read from LDS ahead of their use
#pragma unroll
  for (int i = 0; i < RING; ++i)
    if (P > 0) ring[i] = parked[i * 64];

  // ---- gates: [matrix][16 rows], matrix 0 J1; those past a_dim are not looked at.  (Rows past B: zero; threads without a gate
  // read past the end and write to a spare word.) ----
  const int grow = tid / k, gch = tid - grow * k;
  const unsigned goff = grow < 16 ? (unsigned)(grow * T * k + gch) * 4 : NOWHERE;
  const int gput = grow < 16 ? (1 + gch) * 16 + grow : 2 * S::MATS * 16, gstep = grow < 16 ? S::MATS * 16 : 0;
  auto gate_put = [&](int buf, float v) { gl[gput + buf * gstep] = v; };
  if (tid < 32) gl[((tid >> 4) * S::MATS) * 16 + (tid & 15)] = c.J1;
  // (the tile's buffer ends with the batch; the step is the scalar offset, which is not part of what is checked against its end)
  const int last_bt = c.nbt - 1, rows_last = B - 16 * last_bt;
  const char* const a_first = reinterpret_cast<const char*>(c.A + (size_t)16 * rg * T * k);
  ChipCursor gc{0, 0, a_first, a_first};
  const unsigned a_tile = (unsigned)c.nrg * 16u * (unsigned)T * (unsigned)k * 4u, a_row = (unsigned)T * (unsigned)k * 4u;
  auto gate_of = [&] {
    const bool part = rg + c.nrg * gc.j == last_bt;
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(gc.at), 0, (int)((part ? rows_last : 16) * a_row), 0x00020000);
    const unsigned g = __builtin_amdgcn_raw_buffer_load_b32(ar, (int)goff, gc.t * k * 4, 0);
    return __builtin_bit_cast(float, g);
  };
  gate_put(0, gate_of());
  constexpr int AHEAD = DEPTH < 2 ? 2 : DEPTH;               // items that gates are fetched ahead
  auto gate_fetch = [&] {
    if (gc.t + 1 < T || gc.j + 1 < my_nt) gc.advance(my_nt, a_tile, 0);       // (behind the last item: its own again, unused)
    return gate_of();
  };
  float g0 = gate_fetch(), g1 = gate_fetch(), g2 = AHEAD > 2 ? gate_fetch() : 0.f;

  if (tid == 0) {
    const long long start = wall_clock64();
    bool ok = false;
    unsigned long long v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (!(v & CHIP_GAVE_UP)) {
      if (v == (unsigned long long)c.G) {
        ok = true;
        break;
      }
      if (wall_clock64() - start > c.gather_ticks) {
        // (fails, and leaves the new value in v, if another member has arrived meanwhile)
        if (__hip_atomic_compare_exchange_strong(word, &v, v | CHIP_GAVE_UP, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        continue;
      }
      __builtin_amdgcn_s_sleep(1);
      v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    *reinterpret_cast<int*>(lds + L.go) = ok;
  }
  lds_barrier();
  if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(lds + L.go)) == 0) return;

  // ---- the time loop over items (step, tile) ----
  ChipOperandAt oa;
  const bool in_batch = c.nbt > 1 || b < B;         // (of a single tile only the batch's rows are read)
  oa.x = in_batch ? (unsigned)w * CHUNK_BYTES + lane * 16 : NOWHERE;
  oa.rs = in_batch ? (unsigned)w * CHUNK_BYTES + 1024 + b * 16 + q * 4 : NOWHERE;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool inside = w + W * (KPW - 2 + i) < c.KC;
    oa.x_last[i] = inside ? oa.x : NOWHERE;
    oa.rs_last[i] = inside ? oa.rs : NOWHERE;
  }
  const float oma = 1.f - c.alpha;
  bool dead = c.spin_max < 0;      // (a negative limit gives up at once: the host's way to exercise this exit)
  if (dead && lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
  int it = 0;
  const char* const h_first = reinterpret_cast<const char*>(c.hist + (size_t)16 * rg * N);
  ChipCursor hc{0, 0, h_first, h_first};                                    // the item's history rows
  const size_t h_tile = (size_t)c.nrg * 16 * N * 4, h_step = (size_t)B * N * 4;
  const unsigned x_tile = (unsigned)c.nrg * tile_bytes, x_first = (unsigned)rg * tile_bytes, x_end = (unsigned)c.slots * slot_bytes;
  int load_j = 0;                        // the item whose operand is asked for next
  unsigned load_row = x_first, load_at = x_first;
  ChipOperand<KPW> op[DEPTH];
  auto ask = [&](ChipOperand<KPW>& o) {
    o.issue(rsrc, oa, load_at);
    const bool wrap = load_j + 1 == my_nt;
    const unsigned row = load_row + slot_bytes < x_end ? load_row + slot_bytes : x_first;
    load_row = wrap ? row : load_row;
    load_at = wrap ? row : load_at + x_tile;
    load_j = wrap ? 0 : load_j + 1;
  };
#pragma unroll
  for (int i = 0; i < (DEPTH < 2 ? 1 : DEPTH - 1); ++i) ask(op[i]);

  unsigned at = x_first, at_row = x_first;                                  // its operand
  auto item = [&](ChipOperand<KPW>& now, ChipOperand<KPW>& nx, float& g) {
    if (__builtin_expect(!dead && !now.ready(), 0)) {
      int spins = 0;
      do {
        if (++spins > c.spin_max) {
          dead = true;
          if (lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
        }
        __builtin_amdgcn_s_sleep(1);
        now.issue(rsrc, oa, at);
      } while (!dead && !now.ready());
    }
    gate_put((it + 1) & 1, g);             // the next item's gates, fetched AHEAD items ago
    g = gate_fetch();
    if constexpr (DEPTH > 1) ask(nx);

    bf16x8 xf[KPW];
    float rsum = 0.f;
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) {
      xf[kk] = __builtin_bit_cast(bf16x8, now.x[kk]);
      rsum += __builtin_bit_cast(float, now.rs[kk]);
    }
    const float j0r = c.J0 * sum_bits45(rsum);
    const float* const gates = gl + (it & 1) * S::MATS * 16 + b;
    // sums over the even (0) and the odd matrices; with eight neurons the lane's half of the column tile says which it has
    f32x4 sum[HALVES][2], prod[2];
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sum[h][0][e] = NPW == 8 && q >= 2 ? 0.f : j0r;
        sum[h][1][e] = 0.f;
      }
    auto matrix = [&](int ct) { return NPW == 8 ? 2 * ct : (NPW == 16 ? ct : ct >> 1); };
    float gm[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) gm[ct] = gates[(NPW == 8 ? matrix(ct) + (q >> 1) : matrix(ct)) * 16];
    auto gate_in = [&](int ct) {                                // (behind the next column tile's products)
      const int m0 = matrix(ct), m = NPW == 8 ? m0 + (q >> 1) : m0;
      f32x4& s = sum[NPW == 32 ? ct & 1 : 0][NPW == 8 ? 0 : m0 & 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float with = fmaf(gm[ct], prod[ct & 1][e], s[e]);
        s[e] = ct < S::FULL || m <= k ? with : s[e];            // (nothing of a matrix that is not there, not even of an infinite state)
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    auto products = [&](int ct) {
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk) {
        const int f = ct * KPW + kk, at = S::before(f);
        if (S::is_parked(f)) {
          v = mfma16(ring[at % RING], xf[kk], v);
          ring[at % RING] = parked[(at + RING < P ? at + RING : at % RING) * 64];       // (the first ones for the next item)
        } else {
          v = mfma16(wreg[S::is_parked(f) ? 0 : f - at], xf[kk], v);
        }
      }
      prod[ct & 1] = v;
    };
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      products(ct);
      if (ct > 0) gate_in(ct - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    gate_in(CT - 1);
    float* const put = share + (size_t)((it & 1) * W + w) * S::SHARE + q * CHIP_QS + b * 4;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = NPW == 8 ? sum_bit5(sum[h][0][e]) : sum[h][0][e] + sum[h][1][e];
      if (NPW != 8 || lane < 32) *reinterpret_cast<f32x4*>(put + h * 4 * CHIP_QS) = v;
    }
    lds_barrier();                                              // the item's shares and the next one's gates are in LDS

    // the slots behind and in front of this step's
    const unsigned to_row = at_row + slot_bytes < x_end ? at_row + slot_bytes : x_first, in_row = at - at_row;
    const unsigned to = to_row + in_row, old = (at_row == x_first ? x_end - slot_bytes + x_first : at_row - slot_bytes) + in_row;
    const bool wrap = hc.j + 1 == my_nt, part = rg + c.nrg * hc.j == last_bt;
    const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(hc.at), 0, (part ? rows_last : 16) * N * 4, 0x00020000);
    const float* src = share + (size_t)(it & 1) * W * S::SHARE + (has_out ? (on >> 2) * CHIP_QS + orow * 4 + (on & 3) : 0);
    float* const st = my_state + hc.j * 64 * W;
    float a[W];
#pragma unroll
    for (int v = 0; v < W; ++v) a[v] = src[v * S::SHARE];
    const float r = *st;
#pragma unroll
    for (int v = 1; v < W; ++v) a[0] += a[v];
    const float F_ = chip_act(c.act, a[0]), rn = oj < N ? fmaf(c.alpha, F_, oma * r) : 0.f;
    __builtin_amdgcn_raw_buffer_store_b32(published(rn), rsrc, (int)xoff, (int)to, ST_THROUGH);
    *st = rn;
    __builtin_amdgcn_raw_buffer_store_b32(EMPTY, rsrc, (int)xoff, (int)old, ST_THROUGH);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, rn), hr, (int)hoff, 0, 0);
    if constexpr (DEPTH == 1) {
      // (the first waves' polling would hold up the last ones' stores; also where other groups have two tiles: N = 968, 6 channels,
      // B = 69, T = 40 265 -> 199 us a call)
      if (my_nt == 1) lds_barrier();
      ask(nx);
    }
    ++it;
    hc.advance(my_nt, h_tile, h_step);
    at = wrap ? to_row : at + x_tile;
    at_row = wrap ? to_row : at_row;
  };
  while (hc.t < T) {
    item(op[0], op[DEPTH - 1], g0);
    if (hc.t >= T) break;
    item(op[1 % DEPTH], op[0], g1);
    if constexpr (AHEAD > 2) {
      if (hc.t >= T) break;
      item(op[2 % DEPTH], op[1 % DEPTH], g2);
    }
  }
}

// Eight consecutive neurons of a row of N; past the end: zero.
template <bool WHOLE>
__device__ __forceinline__ void row_eight(const float* row, int N, int j, f32x4& lo, f32x4& hi) {
  if constexpr (WHOLE) {                  // (N is a multiple of four)
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, a = *reinterpret_cast<const f32x4*>(row + (j < N ? j : 0)), b = *reinterpret_cast<const f32x4*>(row + (j + 4 < N ? j + 4 : 0));
    lo = j < N ? a : zero;
    hi = j + 4 < N ? b : zero;
  } else {
    lo = row_quad(row, N, j);
    hi = row_quad(row, N, j + 4);
  }
}

// The tiles of row groups that gave up, on as many workgroups as there are compute units free, with every sum in the order of the
// kernel above.  A unit of work is a step of RT tiles and 16 neurons; workgroups draw units in the order of their steps and wait
// for the step before of the same tiles.  Whoever is waited for has drawn earlier and is running, so this ends with any number of
// workgroups resident, one included.  Weights come from memory for every unit (fp32, read while the wait lasts), the state from the
// history.  A unit's wave w contracts its chunks w, w + 8, ... of all matrices; the eight shares meet in LDS.
template <int KPW, int RT>
__global__ __launch_bounds__(64 * W) void ring_chip_rest_kernel(RingChipArgs c) {
  __shared__ f32x4 share[W][RT][64];
  __shared__ unsigned long long drawn;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4, b = lane & 15;
  const unsigned long long word = __hip_atomic_load(c.gather + (size_t)(lane < c.nrg ? lane : 0) * RING_TEAM_WORD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned groups = (unsigned)__ballot(lane < c.nrg && (word & CHIP_GAVE_UP));
  if (groups == 0) return;
  const int N = c.N, B = c.B, T = c.T, k = c.k;
  const int blocks = (c.nt + RT - 1) / RT, ncg = (N + 15) / 16;                 // tile blocks of a group, column groups
  const unsigned long long per_step = (unsigned long long)__popc(groups) * blocks * ncg, total = per_step * T;
  unsigned long long* const rest = c.gather + (size_t)c.nrg * RING_TEAM_WORD;
  const float oma = 1.f - c.alpha;
  bool dead = c.spin_max < 0;
  if (dead && tid == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
  auto units = [&](auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    for (;;) {
      if (tid == 0) drawn = __hip_atomic_fetch_add(rest, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      const unsigned long long u = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(drawn >> 32)) << 32 |
                                   (unsigned)__builtin_amdgcn_readfirstlane((int)drawn);
      if (u >= total) return;
      const int t = (int)(u / per_step), in_step = (int)(u % per_step), block = in_step / ncg, cg = in_step % ncg;
      unsigned left = groups;
      for (int i = block / blocks; i > 0; --i) left &= left - 1;
      const int rg = __ffs(left) - 1, first = block % blocks * RT;
      auto tile = [&](int i) { return rg + c.nrg * (first + i); };
      unsigned long long* const done = rest + (size_t)(1 + block) * RING_TEAM_WORD;

      WeightLoad l[KPW];
      auto chunk = [&](int kk) {
        int k0 = 32 * (w + W * kk) + 8 * q;
        asm volatile("" : "+v"(k0));         // (or addresses and masks are kept from one matrix to the next: registers)
        return k0;
      };
      auto load = [&](int m) {
        const float* W_ = m == 0 ? c.Wo : c.Wa + (size_t)(m - 1) * N * N;
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk) weight_load<WHOLE ? WEIGHT_ROWS4 : WEIGHT_ROWS>(l[kk], W_, N, 16 * cg + b, chunk(kk));
      };
      load(0);
      if (t > 0) {
        if (tid == 0 && !dead) {
          const unsigned long long want = (unsigned long long)t * ncg;
          for (int spins = 0; __hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want; ++spins) {
            if (spins > c.spin_max) {
              dead = true;
              *c.host_err = RING_CLUSTER_ERR_WAIT;
              break;
            }
            __builtin_amdgcn_s_sleep(8);
          }
        }
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      const float* const prev = t == 0 ? c.r_init : c.hist + (size_t)(t - 1) * B * N;
      bf16x8 x[RT][KPW];
      f32x4 sum[RT][2];                     // the even and the odd matrices
      const float* gates[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int row = 16 * tile(i) + b;
        const size_t at = row < B ? row : B - 1;
        gates[i] = c.A + (at * T + t) * k;
        float rsum = 0.f;
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk) {
          f32x4 lo, hi;
          row_eight<WHOLE>(prev + at * N, N, chunk(kk), lo, hi);
          if (row >= B) lo = hi = f32x4{0.f, 0.f, 0.f, 0.f};
          x[i][kk] = __builtin_bit_cast(bf16x8, u32x4{not_empty(pack_bf16(lo[0], lo[1])), not_empty(pack_bf16(lo[2], lo[3])),
                                                      not_empty(pack_bf16(hi[0], hi[1])), not_empty(pack_bf16(hi[2], hi[3]))});
          rsum += __builtin_bit_cast(float, not_empty(__builtin_bit_cast(unsigned, sum4(lo) + sum4(hi))));
        }
        const float j0r = c.J0 * sum_bits45(rsum);
        sum[i][0] = f32x4{j0r, j0r, j0r, j0r};
        sum[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      auto matrix = [&](int m, int odd) {
        bf16x8 f[KPW];
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk) f[kk] = weight_fragment(l[kk], N, 16 * cg + b, chunk(kk), 1.f, 0.f);
        float g[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) g[i] = m == 0 ? c.J1 : gates[i][m > 0 ? m - 1 : 0];
        if (m < k) load(m + 1);
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          f32x4 P = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < KPW; ++kk) P = mfma16(f[kk], x[i][kk], P);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[i][odd][e] = fmaf(g[i], P[e], sum[i][odd][e]);
        }
      };
#pragma unroll 1
      for (int m = 0; m <= k; m += 2) {
        matrix(m, 0);
        if (m < k) matrix(m + 1, 1);
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) share[w][i][lane] = sum[i][0] + sum[i][1];
      __syncthreads();
      if (w < RT && 16 * tile(w) + b < B) {
        f32x4 v = share[0][w][lane];
        for (int i = 1; i < W; ++i) v += share[i][w][lane];
        const size_t row = 16 * tile(w) + b;
        const int j = 16 * cg + 4 * q;
        const f32x4 r = row_quad(prev + row * N, N, j);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j + e < N)
            __hip_atomic_store(c.hist + ((size_t)t * B + row) * N + j + e, fmaf(c.alpha, chip_act(c.act, v[e]), oma * r[e]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // The stores above go through to where all XCDs see them; here they have arrived.  (Plain stores and a fence, which writes the
      // whole L2 back for every unit: N = 776, 6 channels, B = 656 208 against 71 us per step.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  if ((N & 3) == 0) units(std::true_type{});
  else units(std::false_type{});
}

// ------------------------------------------------------------------------------------------------
// Choice of shape, launch
// ------------------------------------------------------------------------------------------------
// Shapes that are built: neurons per member, K chunks of a wave, column tiles.
#define RING_CHIP_COLUMNS(X, KPW) \
  X(8, KPW, 2) X(8, KPW, 4) X(8, KPW, 7) X(16, KPW, 4) X(16, KPW, 7) X(32, KPW, 6)
// (16, 3, 3: the teams take every call of one or two channels that it has LDS for)
#define RING_CHIP_SHAPES(X)                                                                                          \
  RING_CHIP_COLUMNS(X, 3) X(8, 3, 9) X(32, 3, 8) RING_CHIP_COLUMNS(X, 4) X(8, 4, 9) X(16, 4, 3) X(32, 4, 8)          \
  RING_CHIP_COLUMNS(X, 6) X(8, 6, 9) X(16, 6, 3) X(32, 6, 8) RING_CHIP_COLUMNS(X, 8) X(16, 8, 3)

namespace {

struct ChipRow { int npw, kpw, ct, least, mats, parked[3]; bool built[3]; };      // parked, built: by depth - 1
const ChipRow kChipRows[] = {
#define RING_CHIP_ROW(NPW, KPW, CT)                                                                                                        \
  {NPW, KPW, CT, ChipShape<NPW, KPW, CT, 1>::LEAST, ChipShape<NPW, KPW, CT, 1>::MATS,                                                      \
   {ChipShape<NPW, KPW, CT, 1>::P, ChipShape<NPW, KPW, CT, 2>::P, ChipShape<NPW, KPW, CT, 3>::P},                                          \
   {ChipShape<NPW, KPW, CT, 1>::BUILT, ChipShape<NPW, KPW, CT, 2>::BUILT, ChipShape<NPW, KPW, CT, 3>::BUILT}},
    RING_CHIP_SHAPES(RING_CHIP_ROW)
#undef RING_CHIP_ROW
};

struct ChipPlan {
  bool ok;
  ChipRow row;
  int depth, KC, G, nrg, nt, slots;
  size_t xchg_bytes, gather_bytes;
  float cycles;          // what the model expects of a step
  int rest_tiles() const { return row.kpw > 4 ? 2 : 4; }       // of a tile block of ring_chip_rest_kernel
};

// How long a row group gathers: about what the way round it costs.  us a call, here / all groups given up / panel kernels: N = 2048, 12
// channels, B = 1, T = 60 311 / 3615 / 1429; N = 1100, 2 channels, B = 256, T = 60 487 / 3343 / 887; N = 776, 6 channels, B = 656, T = 20
// 342 / 1429 / 575.  (A workgroup per tile on its own took 1.37 s, 69 ms and 38 ms, and the gathering 50 ms before that.)
constexpr int CHIP_GATHER_US = 5000;

// The kernel goes from a tile's gates to those of the group's next one in 32 bits.
constexpr bool chip_gates_in_reach(int nrg, int T, int k) { return (size_t)nrg * 16 * T * k * 4 <= 0xFFFFFFFFu; }
static_assert(chip_gates_in_reach(8, (1 << 23) - 1, 1) && !chip_gates_in_reach(8, 1 << 23, 1) && !chip_gates_in_reach(8, 1 << 20, 8), "");

ChipPlan chip_plan(int N, int k, int T, int B) {
  ChipPlan best{};
  if (N <= 512 || N > 2048 || k < 1 || k > 16 || B < 1 || T < 1 || (size_t)16 * T * k * 4 >= ((size_t)1 << 30)) return best;
  const int KC = (N + 31) / 32, nbt = (B + 15) / 16;
  int kpw = 0;
  for (const ChipRow& r : kChipRows)
    if (r.kpw * W >= KC && (kpw == 0 || r.kpw < kpw)) kpw = r.kpw;
  const char* force = getenv("RINGATTR_CHIP");           // 8, 16 or 32: neurons per member (cross-checks)
  const int npw = force ? atoi(force) : 0;
  for (const ChipRow& r : kChipRows) {
    if (r.kpw != kpw || r.least > k + 1 || r.mats < k + 1) continue;
    if (npw > 1 && r.npw != npw) continue;
    const int G = 32 * KC / r.npw;                       // (whole K chunks: the padding is published too)
    int nrg = 8;
    while (nrg > 1 && (G > 32 * (8 / nrg) || nrg > nbt)) nrg /= 2;
    if (G > 32 * (8 / nrg)) continue;
    if (!chip_gates_in_reach(nrg, T, k)) continue;
    const int nt = (nbt + nrg - 1) / nrg, slots = nt == 1 ? 8 : (nt < 4 ? 6 : 4);
    const size_t xbytes = (size_t)slots * nbt * KC * CHUNK_BYTES;
    if (xbytes >= ((size_t)1 << 30)) continue;           // (offsets past the buffer say 'nowhere')
    // The deepest prefetch that registers and LDS have room for and the tiles can use: an operand is the state that the group made
    // its tiles' number of items ago, and asked for right behind that item it is not there.  Asking again then holds up the stores it
    // waits for.  us a call of T = 40 with three, two and one operands on their way: three tiles per group, N = 1021, 3 channels,
    // B = 377 539, 261, 279, N = 896, 16 channels, B = 89 404, 239, 266; two tiles, N = 768, 6 channels, B = 121 two and one 225, 150;
    // four, N = 896, B = 121 280, 294, 347.  Where four tiles are the most, a group with three decides for all: B = 107 368, 303.
    const int fewest = nbt / nrg;
    int depth = fewest >= 4 ? 3 : (nt >= 3 ? 2 : 1);
    while (depth > 1 && (depth == 3 ? r.parked[2] > 0 : chip_lds(r.npw, r.mats, r.parked[1], nt).total > CHIP_LDS)) --depth;
    if (!r.built[depth - 1] || chip_lds(r.npw, r.mats, r.parked[depth - 1], nt).total > CHIP_LDS) continue;
    // Cycles of a step at 2.4 GHz, fitted to 180 measured shapes (N = 640 to 2048, 2 to 16 channels, B = 1 to 1024).  Many tiles per
    // group: what an item takes.  One: products, hand-over (the more members, the slower) and epilogue one after the other;
    // a few: the items of a tile wait for its hand-over.
    const int parked = r.parked[depth - 1];
    const float F = (float)(r.ct * r.kpw), kc = (float)KC;
    const float item = 2000.f + 30.f * kc + 25.f * F + (depth == 1 && nt > 2 ? 1100.f : 0.f) + 40.f * (float)parked;
    const float one = 5000.f + 45.f * kc + 25.f * (float)G + 38.f * F - (B < 16 ? 1500.f : 0.f);
    const float cycles = nt == 1 ? one : std::max(1.6f * one, (float)nt * item);
    if (!best.ok || cycles < best.cycles) {
      best = ChipPlan{true, r, depth, KC, G, nrg, nt, slots, (xbytes + 255) & ~(size_t)255, 0, cycles};
      best.gather_bytes = (size_t)(nrg + 1 + nrg * ((nt + best.rest_tiles() - 1) / best.rest_tiles())) * RING_TEAM_WORD * sizeof(unsigned long long);
    }
  }
  return best;
}

}  // namespace

// Where it runs: where the model above expects it to be faster than the step-per-launch kernels, with all channels driven and, within a
// tenth, with two of them.  us per step (T = 60, all channels driven, panel kernels / here; *: stays with the panels as slower,
// +: because of what two driven channels would cost):
//   N = 640,   6 channels: B = 1: 7.4 / 3.1    B = 64: 8.1 / 4.4    B = 1024: 28 / 20 +
//   N = 1024, 16 channels: B = 1: 12.5 / 3.8   B = 32: 12.7 / 5.5   B = 256: 19 / 14 +   B = 1024: 49 / 50 *
//   N = 1100,  2 channels: B = 1: 7.2 / 3.2    B = 64: 9.1 / 5.0    B = 1024: 33 / 28
//   N = 1500, 16 channels: B = 1: 18 / 4.7     B = 64: 20 / 11.5 +  B = 256: 33 / 42 *
//   N = 2048,  2 channels: B = 1: 8.0 / 3.9    B = 64: 10.2 / 6.4   B = 1024: 38 / 44 *;   12 channels, B = 1: 24 / 5.2
// Channels that are silent in all rows of a workgroup (zero-padded action signals) cost the panels nothing; here passing them by
// costs the others more than it saves (N = 1024, B = 1024: 16 channels 49.6 -> 53.6, two of 16 driven 44, panels 22).  What channels
// carry is not known when the kernels are chosen, so the rule protects padded calls, at the price of dense ones as marked.  Of 760
// random calls that it takes (all channels driven or two; T = 60) 15 are slower than on the panels, by 18 % at most (N = 1848, 4
// channels, two driven, B = 124); the mean is 1.74 times as fast.
// Short sequences stay with the panels, whose bits are those of the kernels that write a record: fewer than ten steps gain
// little (loading the weights takes as long as four of them).
static bool chip_rule(const ChipPlan& p, int N, int k, int T, int B) {
  const char* v = getenv("RINGATTR_CHIP");
  if (!p.ok || (v && v[0] == '0') || ring_team_fwd_bytes(N, k, T, B)) return false;       // (teams come first)
  if (v) return true;
  const int NC = (N + 511) / 512 * 8;
  auto panel = [&](int channels) { return ring_panel_step_cycles(NC < 16 ? 16 : NC, (B + 15) / 16, channels); };
  return T >= 10 && p.cycles < 0.95f * panel(k) && p.cycles < 1.1f * panel(k < 2 ? k : 2);
}

bool ring_uses_chip(int N, int k, int T, int B) {
  for (const char* name : {"RINGATTR_PANEL", "RINGATTR_PANEL_SHAPE", "RINGATTR_WIDE", "RINGATTR_BLOCK", "RINGATTR_BLOCK_SHAPE"})
    if (getenv(name)) return false;
  return ring_teams_allowed() && chip_rule(chip_plan(N, k, T, B), N, k, T, B);
}

size_t ring_chip_bytes(int N, int k, int T, int B) {
  const ChipPlan p = chip_plan(N, k, T, B);
  return chip_rule(p, N, k, T, B) ? p.xchg_bytes + p.gather_bytes : 0;
}

template <int NPW, int KPW, int CT, int DEPTH>
static hipError_t chip_start(const RingChipArgs& c, const ChipPlan& p, hipStream_t st) {
  const unsigned dyn = std::max(chip_lds(NPW, p.row.mats, p.row.parked[DEPTH - 1], p.nt).total, 81u * 1024);    // (a compute unit each)
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ring_chip_fwd_kernel<NPW, KPW, CT, DEPTH>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
  if (e != hipSuccess) return e;
  const int per = 8 / p.nrg;
  // (a group that is not complete can hold all of an XCD but one)
  const RingLaunchGuard::Launch order(ring_launch_guard(), st, 31);
  RING_LAUNCH((ring_chip_fwd_kernel<NPW, KPW, CT, DEPTH>), dim3(8u * (unsigned)((p.G + per - 1) / per)), dim3(64 * W), dyn, st, c);
  return hipGetLastError();
}

template <int NPW, int KPW, int CT>
static hipError_t chip_shape(const RingChipArgs& c, const ChipPlan& p, hipStream_t st) {
  if constexpr (ChipShape<NPW, KPW, CT, 3>::BUILT)
    if (p.depth == 3) return chip_start<NPW, KPW, CT, 3>(c, p, st);
  if constexpr (ChipShape<NPW, KPW, CT, 2>::BUILT)
    if (p.depth == 2) return chip_start<NPW, KPW, CT, 2>(c, p, st);
  if constexpr (ChipShape<NPW, KPW, CT, 1>::BUILT)
    if (p.depth == 1) return chip_start<NPW, KPW, CT, 1>(c, p, st);
  return hipErrorInvalidValue;
}

hipError_t ring_chip_fwd(const RingFwdArgs& a, const float* Wo, const float* Wa, void* ws, hipStream_t st) {
  const ChipPlan p = chip_plan(a.N, a.k, a.T, a.B);
  if (!p.ok || !ws || a.dfrag || a.rfrag) return hipErrorInvalidValue;
  RingChipArgs c = {};
  hipError_t e = ring_cluster_host_err(&c.host_err);
  if (e != hipSuccess) return e;
  c.A = a.A;
  c.Wo = Wo;
  c.Wa = Wa;
  c.r_init = a.r_init;
  c.hist = a.hist;
  c.xchg = ws;
  c.xchg_bytes = (unsigned)p.xchg_bytes;
  c.gather = reinterpret_cast<unsigned long long*>(static_cast<char*>(ws) + p.xchg_bytes);
  c.J0 = a.J0;
  c.J1 = a.J1;
  c.alpha = a.alpha;
  c.N = a.N;
  c.k = a.k;
  c.T = a.T;
  c.B = a.B;
  c.nbt = a.nbt;
  c.KC = p.KC;
  c.G = p.G;
  c.nrg = p.nrg;
  c.nt = p.nt;
  c.slots = p.slots;
  c.act = a.act;
  ring_team_limits(&c.spin_max, &c.gather_ticks);
  if (!getenv("RINGATTR_TEAM_GATHER_US")) c.gather_ticks = CHIP_GATHER_US * 100;
  e = ring_team_fill(ws, p.xchg_bytes, p.gather_bytes, st);
  if (e != hipSuccess) return e;
  e = hipErrorInvalidValue;
#define RING_CHIP_CASE(NPW, KPW, CT) \
  if (p.row.npw == NPW && p.row.kpw == KPW && p.row.ct == CT) e = chip_shape<NPW, KPW, CT>(c, p, st);
  RING_CHIP_SHAPES(RING_CHIP_CASE)
#undef RING_CHIP_CASE
  if (e != hipSuccess) return e;
  const int units = p.nrg * ((p.nt + p.rest_tiles() - 1) / p.rest_tiles()) * ((a.N + 15) / 16);
  const dim3 grid((unsigned)std::min(units, 256)), block(64 * W);
  switch (p.row.kpw) {
    case 3: hipLaunchKernelGGL((ring_chip_rest_kernel<3, 4>), grid, block, 0, st, c); break;
    case 4: hipLaunchKernelGGL((ring_chip_rest_kernel<4, 4>), grid, block, 0, st, c); break;
    case 6: hipLaunchKernelGGL((ring_chip_rest_kernel<6, 2>), grid, block, 0, st, c); break;
    case 8: hipLaunchKernelGGL((ring_chip_rest_kernel<8, 2>), grid, block, 0, st, c); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
