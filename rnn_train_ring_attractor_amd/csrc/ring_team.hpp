// Time loops (forward and BPTT) over teams of workgroups: the weights stay on chip, spread by output neuron over the
// workgroups of a team, and the state travels between them through L2 once per step.
//
// What bounds a small or medium batch is not arithmetic but one step's latency: a workgroup that owns its batch rows
// alone has to pull (1 + a_dim) N^2 weights through one compute unit per step (20 us at N = 512) while most of the chip
// idles.  A team of G workgroups on ONE XCD (one L2) splits the N output neurons: member m keeps the rows of
// [Wo | Wa] for its C = 16 * C16 neurons in registers (and, with many channels, LDS) for the whole sequence, so a step
// costs its share of the products plus one hand-over through L2 (a store becomes visible to a sibling's load after
// some 550 cycles on one XCD, 1450 across XCDs, measured).
//
// One item of work is (step, batch tile of 16 rows).  Per item a workgroup's waves have two roles:
//   * WK compute waves split the contraction: wave w owns K chunks w, w + WK, ... (32 neurons each).  It loads just
//     those chunks of the exchanged state, ready made as MFMA operands, multiplies them with its resident weight
//     fragments (weights are the A operand, so a lane ends up with four consecutive neurons of ONE batch row and a
//     gate is one scalar per lane), gates and sums over the matrices in fp32, and leaves its share in LDS.
//   * 4 auxiliary waves add the WK shares in wave order, apply the activation (or form g), publish the new state and
//     write everything that goes to HBM; they also fetch gates, grad_output and the derivative record two items
//     ahead.  The compute waves never wait for HBM: the memory counter is in order, and a wave that had an HBM load
//     in flight could not look at the exchanged state before that load had landed.
// With more than one tile per team the products of an item overlap the epilogue of the item before.
//
// Exchange protocol.  The buffer has `slots` slots, one per state number modulo their count, all of it filled with 0xFF
// before the launch.  A published dword is never 0xFFFFFFFF (a pair of bf16 NaNs that no arithmetic gives;
// publishing clamps it away), so a reader polls the data itself: no flag, no acknowledgement to wait for.  The slot of
// state s - 1 is refilled by its owner in the epilogue of step s: by then every member has published state s, i.e.
// has read all of state s - 1.  It is written again as state s + slots - 1; a reader polls for that only after it has
// read state s + slots - 2 from the same owner, which must have been published after the refill reached L2.  It was:
// an auxiliary wave issues the refill of an item (step s) before the loads of the next one, waits for those in the third
// item after the refill's, before it publishes anything there, and vector-memory operations complete in order.  In
// rounds of the team's tiles that third item is at most step s + 3 with one tile per team, s + 2 with two, s + 1 from
// three up, and what it publishes is state s + 4, s + 3 or s + 2 at the latest: no later than state s + slots - 2, the
// one that has to come behind the refill, with 8 slots where every team has one tile, 6 where the fullest have two or
// three and others one less, 4 from four tiles up (three in some).  Six slots with one tile and four with three are
// exact: one slot less would not do.
// Besides the bf16 state a chunk carries fp32 row sums of the unrounded state (groups of eight neurons, always summed in
// the order of row_sum8, so that a row's bits do not depend on how wide the members are) for the J0 term.
//
// Placement: workgroups go to XCDs round robin by workgroup index, members of a team are 8 indices apart; every
// workgroup has a compute unit of its own (the grid never exceeds the device).  That the members of a team are resident
// together and share an XCD is checked, not assumed: other work may hold compute units (another stream's or process's
// team launch whose members are as incomplete), or a stream may be kept to some of them.  Every member counts itself in
// the team's word before the time loop.  When all have, they stay until the end and nothing can keep them from finishing;
// a team that does not get there within gather_ticks, or meets on different XCDs, gives up as a whole (one atomic word, so
// all members see the same) and leaves its compute units.  A small launch behind this one (ring_team_solo.hip) does the
// tiles of the teams that gave up, a workgroup each and with the same bits, whatever else runs.
// The waits inside the time loop are bounded too: a wave whose wait runs out leaves a word in host memory, waits for
// nothing from then on and goes through the remaining steps on whatever it finds, so the launch ends by itself; the
// library reports the word on its next call.
#pragma once
#include "ring_common.hpp"
#include "ring_kernels.hpp"

#include <type_traits>

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x3 __attribute__((ext_vector_type(3)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int CHUNK_BYTES = 1024 + 256;       // one K chunk of one tile: 16 rows x 32 neurons bf16, 16 rows x 4 fp32 row sums
constexpr unsigned EMPTY = 0xFFFFFFFFu;
constexpr unsigned NOWHERE = 0x80000000u;     // a buffer offset past every buffer's end: loads give 0, stores are dropped
constexpr int AUX = 4;                        // auxiliary waves
// cache policy bits of the buffer instructions.  (Their volatile bit would make the compiler wait for every access on
// the spot; what keeps a poll from being folded into the one before it is the memory clobber in front of it.)
constexpr int LD_COHERENT = 16;       // sc1: past the vector L1
constexpr int ST_LOCAL = 0;

__device__ __forceinline__ unsigned not_empty(unsigned v) { return v == EMPTY ? 0xFFFFFFFEu : v; }

__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(unsigned, v);
}

__device__ __forceinline__ unsigned dpp_xor1(unsigned x) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false); }
__device__ __forceinline__ unsigned dpp_xor2(unsigned x) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false); }
template <int CTRL>
__device__ __forceinline__ float dpp_ror(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// Sum of eight neurons from the sums of their four pairs.
__device__ __forceinline__ float row_sum8(float s0, float s1, float s2, float s3) { return (s0 + s3) + (s2 + s1); }

// Sum over the four lanes of a 16-lane row that differ in lane bits 2-3; in the first of them the order of row_sum8.
__device__ __forceinline__ float sum_bits23(float v) {
  v += dpp_ror<0x124>(v);   // row_ror:4
  v += dpp_ror<0x128>(v);   // row_ror:8
  return v;
}

// Sum over the lanes that differ in lane bits 4 and 5 (the four 16-lane rows of a wave).
__device__ __forceinline__ float sum_bits45(float v) {
  // (the swaps' results go through named integers: a bit cast straight off a vector element reads element 0)
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned a0 = a[0], a1 = a[1];
  const unsigned w = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1));
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  const unsigned b0 = b[0], b1 = b[1];
  return __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
}

// The quad's four lanes hold rows 4r..4r+3 of the same neurons; on return lane j holds all four rows of ONE neuron.
// Four neurons (x = n0 n1, y = n2 n3 as bf16 pairs): lane j has neuron j.
__device__ __forceinline__ u32x2 quad_rows4(unsigned x, unsigned y, int lane) {
  const unsigned sel = (lane & 1) ? 0x03020706u : 0x05040100u;
  const unsigned e0 = __builtin_amdgcn_perm(dpp_xor1(x), x, sel), e1 = __builtin_amdgcn_perm(dpp_xor1(y), y, sel);
  const bool hi = lane & 2;
  const unsigned recv = dpp_xor2(hi ? e0 : e1);
  return hi ? u32x2{recv, e1} : u32x2{e0, recv};
}
// Two neurons (x = n0 n1): lanes 0, 2 have neuron 0, lanes 1, 3 neuron 1.
__device__ __forceinline__ u32x2 quad_rows2(unsigned x, int lane) {
  const unsigned sel = (lane & 1) ? 0x03020706u : 0x05040100u;
  const unsigned e0 = __builtin_amdgcn_perm(dpp_xor1(x), x, sel);
  const unsigned recv = dpp_xor2(e0);
  return (lane & 2) ? u32x2{recv, e0} : u32x2{e0, recv};
}

// Eight consecutive weights of one output neuron `out`, contraction indices k0 .. k0 + 7, from an fp32 [N][N] matrix.
// Loads and arithmetic are apart so that several fragments' loads can be in flight; addresses are clamped into the
// matrix and the padding is zeroed afterwards.  ROWS4 (rows that start on 16-byte boundaries): two 16-byte loads, eight
// fragments on their way; a call of T = 20 steps at N = 512, 16 channels, B = 256 falls from 181 us (a word at a time, four
// fragments) to 106, at N = 1024, two channels, B = 1 from 105 to 61 (all on their way at once into one XCD: 12.6 MB).
// Other rows are slower so than a word at a time in a team (N = 1023, B = 100: 140 against 98 us).
struct WeightLoad { float v[8]; };
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
enum : int { WEIGHT_ROWS, WEIGHT_ROWS4, WEIGHT_COLUMNS };      // COLUMNS: the transposed matrix

template <int HOW>
__device__ __forceinline__ void weight_load(WeightLoad& l, const float* __restrict__ W, int N, int out, int k0) {
  const unsigned o = out < N ? out : N - 1;
  if constexpr (HOW == WEIGHT_COLUMNS) {
#pragma unroll
    for (int x = 0; x < 8; ++x) l.v[x] = W[(size_t)(k0 + x < N ? k0 + x : N - 1) * N + o];
  } else if constexpr (HOW == WEIGHT_ROWS4) {      // (N is a multiple of four: a group of four is in the row or past it)
    const unsigned at = o * (unsigned)N;             // (32 bits here: one register an address, not two)
    const f32x4 lo = *reinterpret_cast<const f32x4*>(W + (at + (unsigned)(k0 < N ? k0 : 0))),
                hi = *reinterpret_cast<const f32x4*>(W + (at + (unsigned)(k0 + 4 < N ? k0 + 4 : 0)));
#pragma unroll
    for (int x = 0; x < 4; ++x) { l.v[x] = lo[x]; l.v[4 + x] = hi[x]; }
  } else {
#pragma unroll
    for (int x = 0; x < 8; ++x) l.v[x] = W[(size_t)o * N + (k0 + x < N ? k0 + x : N - 1)];
  }
}
__device__ __forceinline__ bf16x8 weight_fragment(const WeightLoad& l, int N, int out, int k0, float scale, float shift) {
  bf16x8 f;
#pragma unroll
  for (int x = 0; x < 8; ++x) f[x] = (__bf16)((out < N && k0 + x < N) ? fmaf(l.v[x], scale, shift) : 0.f);
  return f;
}

// Where an auxiliary thread's outputs of an item live.  NPT consecutive neurons of one row: 16-lane rows hold four
// batch rows x whole 32-byte sectors of everything that is stored.
template <int C16>
struct AuxMap {
  static constexpr int NPT = C16 == 4 ? 4 : 2;
  static constexpr int QS = C16 == 4 ? 80 : 96;      // LDS floats between the q groups of a share (bank spread)
  static constexpr int SHARE = 4 * QS;               // floats of one wave's share of one column tile
  int c, q, p, b;      // column tile of the member, neuron quad, pair inside the quad, row
  bool active;
  __device__ __forceinline__ explicit AuxMap(int at) {
    const int aw = at >> 6, lane = at & 63, s2 = (lane >> 2) & 3;
    b = (lane & 3) | ((lane >> 4) << 2);
    if constexpr (C16 == 4) {
      c = aw;
      q = s2;
      p = 0;
      active = true;
    } else {
      const int s = (aw & 1) * 4 + s2;
      c = aw >> 1;
      q = s >> 1;
      p = s & 1;
      active = c < C16;
      if (!active) c = 0;
    }
  }
};

// K chunk number i in the order of the weight-resident forward's contraction (split_k_neuron): even ones, odd ones.
__host__ __device__ __forceinline__ int rows_chunk(int i) { return 2 * (i & 3) + (i >> 2); }

template <int C16, int WK>
constexpr size_t share_floats() { return (size_t)2 * WK * C16 * AuxMap<C16>::SHARE; }

// The fullest shapes leave a few of a wave's fragments in LDS: with all of them in registers the compiler spills one or
// two, and a reload from scratch memory waits behind the operand prefetch (one in-order counter).
template <int KPW, int C16, int MR, bool GA>
constexpr int parked_fragments() { return KPW * C16 * MR < 24 ? 0 : (GA ? 4 : 2); }
// (a launch reserves for either variant)
inline __host__ __device__ int parked_bytes(int kpw, int c16, int mr, int wk) { return kpw * c16 * mr < 24 ? 0 : wk * 4 * 1024; }

struct LdsPlan {       // byte offsets into dynamic LDS
  unsigned share, state, held, gates, gathered, rows, ga, parked, weights, total;
};

// k: channels; nt: tiles of the fullest team; lds_mats: matrices kept in LDS; KC: K chunks
template <int C16, int WK>
__host__ __device__ inline LdsPlan lds_plan(int k, int nt, int lds_mats, int KC, int parked, bool bptt, bool ga) {
  LdsPlan p;
  unsigned at = 0;
  p.share = at;
  at += (unsigned)share_floats<C16, WK>() * 4;
  p.state = at;
  at += (unsigned)nt * C16 * 256 * 4;
  p.held = at;
  at += bptt ? (unsigned)nt * C16 * 256 * 2 : 0;
  p.gates = at;
  at += ((unsigned)3 * k * 16 + 64) * 4;                  // two buffers, and the spare words of TeamGates::put
  p.gathered = at - 64;
  p.rows = at;                                            // dL/dA: r_prev of the item's rows, this member's neurons
  at += ga ? (unsigned)2 * C16 * 256 * 4 : 0;
  p.ga = at;                                              // dL/dA: shares [2][WK][k][16]
  at += ga ? (unsigned)2 * WK * k * 16 * 4 : 0;
  p.parked = at;
  at += (unsigned)parked;
  p.weights = at;
  at += (unsigned)lds_mats * C16 * KC * 1024;
  p.total = at;
  return p;
}

// ------------------------------------------------------------------------------------------------
// Compute role, shared by forward and BPTT.  EX: matrices in LDS, none, exactly that many, or TEAM_MORE: any number.
// ------------------------------------------------------------------------------------------------
constexpr int TEAM_MORE = 100;

template <int KPW, int C16, int MR, int WK, int EX, bool GA>
struct TeamCompute {
  static constexpr int F = MR * C16 * KPW, FR = F - parked_fragments<KPW, C16, MR, GA>();
  bf16x8 wreg[FR];                 // fragment (matrix, column tile, chunk) in that order
  bf16x8* parked;                  // the lane's slots of the others
  // Lane offsets of an operand fragment and a row sum behind the wave's first chunk; the later chunks are WK apart (scalar
  // offsets).  Only the last one can lie past the contraction: its lanes then point past the buffer and read zero.
  unsigned x_lane, rs_lane, x_last, rs_last;

  // The order of the loads, by what was measured.  Rolling: a fragment's place is loaded again as soon as it is converted.
  // Otherwise batches drain before the next begins.  Rows on 16-byte boundaries roll (in batches the loads' registers spill,
  // 780 bytes a lane in the kernel of 13 matrices in registers, and two calls, N = 512 with 16 channels and N = 1024 with two,
  // take 131 and 74 us, not 106 and 61).  A word at a time, batches of four spill less: us a call, T = 20, rolling and in
  // batches: N = 129, 3 channels, B = 64 33 and 29; N = 513, 3 channels, B = 1 78 and 65; N = 1023, 2 channels, B = 1 94 and 72;
  // training N = 1023, B = 64 227 and 188.  Only with 24 fragments in registers and matrices in LDS do batches leave spills in the
  // loop over the steps, also for rows on 16-byte boundaries (N = 800, 3 channels, B = 300 106 and 134).
  template <int HOW>
  __device__ __forceinline__ void load_matrices(const RingTeamArgs& c, bf16x8* wl, int mem, int w, int lane) {
    constexpr bool ROLL = HOW == WEIGHT_ROWS4 || (EX && F >= 24);
    constexpr int BATCH = HOW == WEIGHT_ROWS4 ? 8 : 4;      // fragments on their way at a time
    const int q = lane >> 4, n = lane & 15;
    auto matrix = [&](int mm) { return mm == 0 || mm > c.k ? c.Wo : c.Wa + (size_t)(mm - 1) * c.N * c.N; };
    // into LDS: the matrices past the registers', this wave's own chunks
    if constexpr (EX) {
      auto load = [&](WeightLoad& l, int mm, int cc, int kc) {
        weight_load<HOW>(l, c.Wa + (size_t)(mm - 1) * c.N * c.N, c.N, 16 * (mem * C16 + cc) + n, 32 * kc + 8 * q);
      };
      auto put = [&](const WeightLoad& l, int mm, int cc, int kc) {
        wl[((size_t)((mm - MR) * C16 + cc) * c.KC + kc) * 64 + lane] = weight_fragment(l, c.N, 16 * (mem * C16 + cc) + n, 32 * kc + 8 * q, 1.f, 0.f);
      };
      if constexpr (ROLL) {
        const int total = (c.k + 1 - MR) * C16 * KPW;
        for (int f0 = 0; f0 < total; f0 += BATCH) {
          WeightLoad l[BATCH];
#pragma unroll
          for (int i = 0; i < BATCH; ++i) {
            const int f = f0 + i < total ? f0 + i : total - 1;
            load(l[i], MR + f / (C16 * KPW), f / KPW % C16, w + WK * (f % KPW));
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < BATCH; ++i) {
            const int f = f0 + i, kc = w + WK * (f % KPW);
            if (f < total && kc < c.KC) put(l[i], MR + f / (C16 * KPW), f / KPW % C16, kc);
          }
        }
      } else {
        for (int mm = MR; mm <= c.k; ++mm)
          for (int kc = w; kc < c.KC; kc += WK) {
            WeightLoad l[C16];
#pragma unroll
            for (int cc = 0; cc < C16; ++cc) load(l[cc], mm, cc, kc);
#pragma unroll
            for (int cc = 0; cc < C16; ++cc) put(l[cc], mm, cc, kc);
          }
      }
    }
    // into registers
    auto load = [&](WeightLoad& l, int f) {
      weight_load<HOW>(l, matrix(f / (C16 * KPW)), c.N, 16 * (mem * C16 + f / KPW % C16) + n, 32 * (w + WK * (f % KPW)) + 8 * q);
    };
    auto keep = [&](const WeightLoad& l, int f) {
      const int mm = f / (C16 * KPW);
      bf16x8 v = weight_fragment(l, mm <= c.k ? c.N : 0, 16 * (mem * C16 + f / KPW % C16) + n, 32 * (w + WK * (f % KPW)) + 8 * q,
                                 mm == 0 ? c.scale0 : 1.f, mm == 0 ? c.shift0 : 0.f);
      asm volatile("" : "+v"(v));          // (converted here, not at its first use: twice the registers until then)
      if (f < FR) wreg[f < FR ? f : 0] = v;
      else parked[(f - FR) * 64] = v;
    };
    if constexpr (ROLL) {
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
    } else {
#pragma unroll
      for (int f0 = 0; f0 < F; f0 += BATCH) {
        WeightLoad l[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
          if (f0 + i < F) load(l[i], f0 + i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
          if (f0 + i < F) keep(l[i], f0 + i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  template <bool TR>
  __device__ __forceinline__ void load_weights(const RingTeamArgs& c, bf16x8* wl, bf16x8* parked_area, int mem, int w, int lane) {
    parked = parked_area + (size_t)w * (F - FR) * 64 + lane;
    const unsigned first = (unsigned)w * CHUNK_BYTES;
    x_lane = first + lane * 16;
    rs_lane = first + 1024 + (lane & 15) * 16 + (lane >> 4) * 4;
    const bool whole = w + WK * (KPW - 1) < c.KC;
    x_last = whole ? x_lane : NOWHERE;
    rs_last = whole ? rs_lane : NOWHERE;
    if constexpr (TR) load_matrices<WEIGHT_COLUMNS>(c, wl, mem, w, lane);
    else if ((c.N & 3) == 0) load_matrices<WEIGHT_ROWS4>(c, wl, mem, w, lane);
    else load_matrices<WEIGHT_ROWS>(c, wl, mem, w, lane);
  }
};

template <int KPW>
struct TeamOperand {
  u32x4 x[KPW];
  unsigned rs[KPW];            // lane (q, row): the row sum over neurons 8q .. 8q + 7 of the chunk
  // (the memory clobber keeps a load from being folded into the same one a poll earlier)
  template <int WK, typename TC>
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rsrc, const TC& tc, unsigned base) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) {
      x[kk] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(kk + 1 < KPW ? tc.x_lane : tc.x_last), (int)(base + kk * WK * CHUNK_BYTES), LD_COHERENT);
      rs[kk] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(kk + 1 < KPW ? tc.rs_lane : tc.rs_last), (int)(base + kk * WK * CHUNK_BYTES), LD_COHERENT);
    }
  }
  __device__ __forceinline__ bool ready() const {
    unsigned m = 0;
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) m = max(max(max(m, rs[kk]), max(x[kk][0], x[kk][1])), max(x[kk][2], x[kk][3]));
    return __ballot(m == EMPTY) == 0;
  }
};

// One item's products: acc[c] = J1 * P_0 + J0 * rowsum + sum_m gate_m P_m over this wave's K chunks: the matrices in registers
// and those in LDS (any number of them: up to channel `last`).
template <int KPW, int C16, int MR, int WK, int EX, bool GA>
__device__ __forceinline__ void team_products(const TeamCompute<KPW, C16, MR, WK, EX, GA>& tc, const TeamOperand<KPW>& op,
                                              const RingTeamArgs& c, const bf16x8* wl, const float (&gate)[MR], const float* gates,
                                              const f32x4* rows, float* ga, int w, int lane, int last, f32x4 (&acc)[C16]) {
  const int b = lane & 15;
  bf16x8 x[KPW];
#pragma unroll
  for (int kk = 0; kk < KPW; ++kk) x[kk] = __builtin_bit_cast(bf16x8, op.x[kk]);
  constexpr int FR = TeamCompute<KPW, C16, MR, WK, EX, GA>::FR;
  auto weight = [&](int f) { return f < FR ? tc.wreg[f < FR ? f : 0] : tc.parked[(f - FR) * 64]; };   // (f is a constant everywhere)
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto row_dot = [&](float& d, const f32x4& P, int cc) {     // dL/dA: this wave's share of sum_j P[j] r_prev[j]
    if constexpr (GA) {
      const f32x4 rp = rows[cc * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) d = fmaf(P[i], rp[i], d);
    }
  };
  auto row_put = [&](float d, int m) {
    if constexpr (GA) {
      d = sum_bits45(d);
      if (lane < 16) ga[(m - 1) * 16 + b] = d;
    }
  };
#pragma unroll
  for (int cc = 0; cc < C16; ++cc) {
    acc[cc] = zero;
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) acc[cc] = mfma16(weight(cc * KPW + kk), x[kk], acc[cc]);
  }
  {
    float rsum = 0.f;
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk) rsum += __builtin_bit_cast(float, op.rs[kk]);
    const float j0r = c.J0 * sum_bits45(rsum);
#pragma unroll
    for (int cc = 0; cc < C16; ++cc)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[cc][i] = fmaf(c.J1, acc[cc][i], j0r);
  }
#pragma unroll
  for (int m = 1; m < MR; ++m) {                 // (channels past a_dim: zero weights and a zero gate)
    float d = 0.f;
#pragma unroll
    for (int cc = 0; cc < C16; ++cc) {
      f32x4 P = zero;
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk) P = mfma16(weight((m * C16 + cc) * KPW + kk), x[kk], P);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[cc][i] = fmaf(gate[m], P[i], acc[cc][i]);
      row_dot(d, P, cc);
    }
    if (GA && m <= c.k) row_put(d, m);
  }
  // The matrices in LDS.  Where their number is known and registers are left (not beside 24 and more fragments: with 13 matrices in
  // registers the reads spill, forward N = 512, 16 channels, B = 256, T = 20 92.6 -> 180 us a call), a matrix's first fragments are read
  // while the one before it is multiplied, the first matrix's behind the registers' products: an LDS read's latency less a matrix.  us a
  // call of T = 40, forward: N = 300, 9 channels, B = 800 278 -> 260; N = 700, 4 channels, B = 500 218 -> 203; N = 360, 3 channels,
  // B = 1000 150 -> 140; N = 144, 3 channels, B = 900 73 -> 68.  Any number of matrices: reads ahead cost what they gain (N = 112, 16
  // channels, B = 200, T = 60 144 -> 151).
  constexpr bool AHEAD = EX != TEAM_MORE && MR * C16 * KPW <= 18;
  bf16x8 f[KPW];
  auto fetch = [&](int m) {
    if constexpr (!AHEAD) return;
    const bf16x8* src = wl + ((size_t)(m - MR) * C16 * c.KC + w) * 64 + lane;
#pragma unroll
    for (int kk = 0; kk < KPW; ++kk)
      if (kk + 1 < KPW || w + WK * kk < c.KC) f[kk] = src[(size_t)WK * kk * 64];
  };
  auto lds_matrix = [&](int m, float gm, int next) {
    bf16x8 f0[KPW];
    if constexpr (AHEAD) {
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk) f0[kk] = f[kk];
      if (next) fetch(next);
    }
    // a channel that is zero for all 16 rows contributes nothing (zero-padded action signals); dL/dA needs every product
    if (!GA && __ballot(gm != 0.f) == 0) return;
    float d = 0.f;
#pragma unroll
    for (int cc = 0; cc < C16; ++cc) {
      f32x4 P = zero;
      const bf16x8* src = wl + ((size_t)((m - MR) * C16 + cc) * c.KC + w) * 64 + lane;
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk)
        if (kk + 1 < KPW || w + WK * kk < c.KC) P = mfma16(AHEAD && cc == 0 ? f0[kk] : src[(size_t)WK * kk * 64], x[kk], P);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[cc][i] = fmaf(gm, P[i], acc[cc][i]);
      row_dot(d, P, cc);
    }
    row_put(d, m);
  };
  if constexpr (EX == TEAM_MORE) {
    // (gates are read a matrix ahead: forward N = 512, 16 channels, B = 256, T = 20 95.5 -> 93.2 us, N = 168, B = 223, T = 76 158.7 -> 152.3)
    float gn = gates[(MR - 1) * 16 + b];
    for (int m = MR; m <= last; ++m) {
      const float gm = gn;
      gn = gates[(m < c.k ? m : c.k - 1) * 16 + b];
      lds_matrix(m, gm, 0);
    }
  } else if constexpr (EX > 0) {
    float g[EX];
#pragma unroll
    for (int i = 0; i < EX; ++i) g[i] = gates[(MR - 1 + i) * 16 + b];
    fetch(MR);
#pragma unroll
    for (int i = 0; i < EX; ++i) lds_matrix(MR + i, g[i], i + 1 < EX ? MR + i + 1 : 0);
  }
}

// Residence of the whole team (see the top of this file).  The first auxiliary wave counts its workgroup in with
// team_arrive, waits in team_gather and leaves the verdict in LDS for all waves to read behind the next barrier (team_go).
constexpr unsigned long long TEAM_GAVE_UP = 1ull << 63;

__device__ __forceinline__ unsigned long long* team_word(const RingTeamArgs& c, int team) { return c.gather + (size_t)team * RING_TEAM_WORD; }
__device__ __forceinline__ int xcc_id() { return __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 7; }
__device__ __forceinline__ unsigned team_arrived(unsigned long long v) { return (unsigned)((v * 0x0101010101010101ull) >> 56); }
__device__ __forceinline__ bool team_complete(unsigned long long v, int G, int xcc) {
  return !(v & TEAM_GAVE_UP) && (int)((v >> (8 * xcc)) & 255) == G;
}

__device__ __forceinline__ void team_arrive(const RingTeamArgs& c, int team, int at) {
  if (at != 0) return;
  if (c.gather_ticks < 0) __hip_atomic_fetch_or(team_word(c, team), TEAM_GAVE_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else __hip_atomic_fetch_add(team_word(c, team), 1ull << (8 * xcc_id()), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void team_gather(const RingTeamArgs& c, char* lds, const LdsPlan& L, int team, int at) {
  if (at != 0) return;
  const int xcc = xcc_id();
  const long long start = wall_clock64();
  bool ok = false;
  unsigned long long v = __hip_atomic_load(team_word(c, team), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (!(v & TEAM_GAVE_UP)) {
    if ((int)team_arrived(v) == c.G) {
      ok = team_complete(v, c.G, xcc);
      if (!ok) __hip_atomic_fetch_or(team_word(c, team), TEAM_GAVE_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    if (wall_clock64() - start > c.gather_ticks) {
      // (fails, and leaves the new value in v, if another member has arrived meanwhile)
      if (__hip_atomic_compare_exchange_strong(team_word(c, team), &v, v | TEAM_GAVE_UP, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        break;
      continue;
    }
    __builtin_amdgcn_s_sleep(1);
    v = __hip_atomic_load(team_word(c, team), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  *reinterpret_cast<int*>(lds + L.gathered) = ok;
}

__device__ __forceinline__ bool team_go(const char* lds, const LdsPlan& L) {
  return __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(lds + L.gathered)) != 0;
}

// When a wave first looks for the next state where a team has one tile.  The state is there some 900 cycles behind the barrier that
// ends the products (sums, activation, a store on its way), a look takes some 450, and one that comes back too early holds up the
// next by as much: looked for before the products, or at once behind them, a step waited up to a whole look too long, the same in every
// step.  So the first look goes out `look` times 64 cycles behind the barrier.  (The time does not fall and rise once with `look`: later
// looks follow the first at fixed distances, and what counts is when the one that finds the state went out.)  us a call, gelu unless
// said, looking before the products (teams of several tiles' way), at once behind the barrier, and 4, 8, 10 and 12 times 64 cycles later:
//   rows kernels, forward, T = 100        0      4      8     10     12        BPTT     0      4      8     10     12
//     N = 256, B = 1                     83.8   92.8   83.7   84.5   88.0             106.4  117.0  104.7  108.7  114.5
//       relu                             82.5   80.1   77.9   82.0   86.9
//     N = 256, B = 8                     89.2   95.7   88.3   89.0   89.5    (4 rows) 107.6  119.2  105.5  108.8  114.5
//     N = 200, B = 8, tanh               84.4   90.0   81.5   83.2   86.9
//     N = 256, B = 16                    94.2  101.8   94.3   93.4   92.3             127.1  139.5  124.3  124.8  125.1
//       relu                             91.5   89.4   86.0   85.3   88.4             124.9  137.4  123.7  123.2  124.8
//     N = 256, B = 128                   95.0  102.6   95.2   93.8   92.8             135.1  147.6  132.6  133.9  133.7
//     N = 200, B = 128                   90.3   98.8   91.4   90.5   90.0             127.5  139.1  126.6  127.1  127.1
//     N = 131, B = 384, tanh             91.3   99.3   89.1   88.9   90.5
//     N = 200, B = 512, tanh (two tiles) 100.0  99.5   96.6   96.0  101.1  (400 rows) 139.3  147.0  136.8  137.7  137.2
//   So 8, and 10 in a forward of more than eight rows.
//   others, T = 60               before   0      4      8     10     12      BPTT before   0      4      8     10     12
//     N = 300, B = 60             71.7   67.8   70.9   66.7   66.5   70.1           98.9   95.5   99.0   94.2   96.6   99.2
//     N = 360, 3 channels, B = 60 80.4   77.7   81.0   75.5   75.4   78.7          109.7  107.6  112.0  106.3  107.8  111.5
//     N = 512, B = 60             81.8   79.1   81.4   75.0   74.4   77.5          115.4  113.1  115.3  109.4  110.3  112.3
//       tanh                      78.5   77.5   74.2   71.0   74.4   77.5
//     N = 600, B = 60            101.4  100.9  102.9   95.7   94.0   93.8          132.2  130.6  132.8  123.4  123.5  123.9
//     N = 800, 3 channels, B = 1 141.2  142.4  141.1  132.7  130.6  130.1          179.3  182.9  183.7  175.2  174.1  178.7
//     N = 1024, B = 60           140.0  141.0  138.1  131.9  128.3  125.1          193.2  189.8  187.9  179.0  178.3  178.7
//       tanh                     135.4  135.0  133.1  123.9  121.6  124.0
//   So 8 up to two chunks a compute wave, past that 12 forward and 10 backward.  (N = 800, 3 channels: the late BPTT spills 92 registers
//   a lane, the other 79, and is ahead all the same: B = 128 223.2, 221.3 with 12 and 219.2 with 10.)
// With many matrices the compute waves are what is waited for, and they look before the products as with several tiles: forward
// N = 512, 16 channels, B = 128, T = 40 108.6  108.1  109.7  111.5; N = 120, 12 channels, B = 30, T = 100 189  192  196  192.
// (lds_mats: or TEAM_MORE.)  Kernels of their own: a second loop in the others', or a branch around their loads, costs those that look
// early (forward N = 400, 9 channels, B = 200, T = 60 132 -> 137 us; training N = 1024, B = 512, T = 40 547 -> 840).
// Four column tiles a member, and two where one fits the matrices as well, are only taken where teams have several tiles.
__host__ __device__ constexpr bool team_may_look_late(int kpw, int c16, int mr, int wk, int lds_mats) {
  return mr == 3 && wk == 8 && lds_mats <= 4 && (c16 == 1 || kpw >= 3 || (c16 == 2 && (kpw == 1 ? lds_mats <= 1 : lds_mats >= 3)));
}
__device__ __forceinline__ void team_look(int look) {
  for (int i = 0; i < look; ++i) __builtin_amdgcn_s_sleep(1);
}

// The compute waves' loop: `steps` rounds over the team's my_nt tiles, operand number s of round s.
// (TR: with the transposed matrices)
template <bool TR, int KPW, int C16, int MR, int WK, int EX, bool GA, bool LATE>
__device__ __forceinline__ void team_compute_loop(const RingTeamArgs& c, const LdsPlan& L, char* lds,
                                                  __amdgpu_buffer_rsrc_t rsrc, int mem, int team, int my_nt, int steps, int w,
                                                  int lane) {
  using AM = AuxMap<C16>;
  constexpr bool PADS = EX == TEAM_MORE && MR == 3 && !GA;             // (dL/dA needs every product)
  TeamCompute<KPW, C16, MR, WK, EX, GA> tc;
  bf16x8* const wl = reinterpret_cast<bf16x8*>(lds + L.weights);
  tc.template load_weights<TR>(c, wl, reinterpret_cast<bf16x8*>(lds + L.parked), mem, w, lane);
  const int q = lane >> 4, b = lane & 15;
  float* const share = reinterpret_cast<float*>(lds + L.share) + (size_t)w * C16 * AM::SHARE + q * AM::QS + b * 4;
  const float* const gates = reinterpret_cast<const float*>(lds + L.gates);
  const f32x4* const rows = reinterpret_cast<const f32x4*>(lds + L.rows);
  float* const ga = reinterpret_cast<float*>(lds + L.ga);
  const unsigned tile_bytes = (unsigned)c.KC * CHUNK_BYTES;
  const unsigned slot_bytes = tile_bytes * (unsigned)c.nbt;
  lds_barrier();                                          // the auxiliary waves' first gates (and rows) are in LDS
  if (!team_go(lds, L)) return;
  TeamOperand<KPW> opA, opB;
  int slot = 0, it = 0, s = 0, j = 0;
  bool dead = c.spin_max < 0;      // (a negative limit gives up at once: the host's way to exercise this exit)
  if (dead && lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
  opA.template issue<WK>(rsrc, tc, (unsigned)team * tile_bytes);
  // One item.  The operand of the next one is fetched meanwhile: with several tiles per team it usually is published
  // already (its state was formed a round ago), with one tile and many matrices this is the first poll for it.  Whether it was there is
  // checked when it is used.  (LATE: one tile, and the next item's operand is asked for at its start.)
  auto item = [&](TeamOperand<KPW>& op, TeamOperand<KPW>& nx) {
    float gate[MR];                  // (in LDS since the last barrier; read while the operand is on its way)
#pragma unroll
    for (int m = 1; m < MR; ++m) gate[m] = m <= c.k ? gates[(it & 1) * c.k * 16 + (m - 1) * 16 + b] : 0.f;
    // Zero-padded action signals: are all channels whose matrices are in LDS silent in the item's rows?  Their gates (up to 14
    // channels of 16 rows) lie one after the other: four a lane, looked at once the operand is there.  Asked matrix by matrix, one
    // read of a gate behind the other, silent channels took a quarter of an item: training N = 112, B = 200, T = 100, 16 channels,
    // two driven 455 -> 325 us a pass.  With nine or thirteen matrices in registers few are left to ask for, and it costs the
    // others: 16 channels, all driven, N = 512, B = 256, T = 20 93.2 us a call, 96.1 with it (two driven: N = 300, B = 500, T = 100,
    // training 1612 and 1479).  A second copy of the products without the silent matrices in registers: 1253, but 8 % more where all
    // are driven.
    u32x4 tail = {1u, 1u, 1u, 1u};
    if (PADS && c.k > MR) {
      const int first = (MR - 1) * 16 + 4 * lane;
      tail = *reinterpret_cast<const u32x4*>(gates + (it & 1) * c.k * 16 + (first < c.k * 16 ? first : (MR - 1) * 16));
    }
    int spins = 0;
    if constexpr (LATE) {                                  // (one tile per team)
      if (s > 0) {
        team_look(c.look);
        op.template issue<WK>(rsrc, tc, (unsigned)slot * slot_bytes + (unsigned)team * tile_bytes);
      }
    }
    // Wide rings: the operand is nearly always there when several tiles share a team, and with the polling loop out of the
    // way the path straight on is shorter: N = 700, B = 500 11.55 -> 11.1 us per step forward and backward, N = 1024,
    // B = 2048 51.2 -> 50.3.  Up to N = 512 it gains nothing (and N = 120, B = 64 in teams of eight loses 2 %).
    if constexpr (KPW >= 3) {
      if (__builtin_expect(!dead && !op.ready(), 0)) {
        const unsigned at = (unsigned)slot * slot_bytes + (unsigned)(team + c.nteams * j) * tile_bytes;
        do {
          if (++spins > c.spin_max) {
            dead = true;
            if (lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
          }
          op.template issue<WK>(rsrc, tc, at);
        } while (!dead && !op.ready());
      }
    } else {
      while (!dead && !op.ready()) {
        if (++spins > c.spin_max) {
          dead = true;
          if (lane == 0) *c.host_err = RING_CLUSTER_ERR_WAIT;
        }
        op.template issue<WK>(rsrc, tc, (unsigned)slot * slot_bytes + (unsigned)(team + c.nteams * j) * tile_bytes);
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0), for the compiler's books: this operand has landed on every path
    const bool wrap = j + 1 == my_nt;
    const int jn = wrap ? 0 : j + 1, sn = !wrap ? slot : (slot + 1 == c.slots ? 0 : slot + 1);
    if constexpr (!LATE) nx.template issue<WK>(rsrc, tc, (unsigned)sn * slot_bytes + (unsigned)(team + c.nteams * jn) * tile_bytes);
    f32x4 acc[C16];
    const bool padding = PADS && __ballot(((tail[0] | tail[1] | tail[2] | tail[3]) & 0x7FFFFFFFu) != 0) == 0;
    team_products<KPW, C16, MR, WK, EX, GA>(tc, op, c, wl, gate, gates + (it & 1) * c.k * 16, rows + (it & 1) * C16 * 64,
                                            ga + (size_t)((it & 1) * WK + w) * c.k * 16, w, lane, padding ? 0 : c.k, acc);
    float* dst = share + (it & 1) * (WK * C16 * AM::SHARE);
#pragma unroll
    for (int cc = 0; cc < C16; ++cc) *reinterpret_cast<f32x4*>(dst + cc * AM::SHARE) = acc[cc];
    lds_barrier();
    ++it;
    j = jn;
    slot = sn;
    s += wrap ? 1 : 0;
  };
  while (s < steps) {
    item(opA, opB);
    if (s >= steps) break;
    item(opB, opA);
  }
}

// ------------------------------------------------------------------------------------------------
// Auxiliary role: pieces shared by forward and BPTT.
// ------------------------------------------------------------------------------------------------
// Every store of the epilogue is a buffer store with one lane-constant offset and a scalar base; what a lane or a step
// has nothing to store for lies past the buffer's end and is dropped there.  No branches, so the compiler knows how
// many memory operations follow a load and waits for that load alone.

__device__ __forceinline__ __amdgpu_buffer_rsrc_t team_buffer(const void* base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(bytes < 0x7FFFFFFFu ? bytes : 0x7FFFFFFFu), 0x00020000);
}

template <int C16>
struct TeamAux {
  using AM = AuxMap<C16>;
  static constexpr int NPT = AM::NPT;
  AM map;
  int at, lane, j0, ct;
  bool tile_ok;                       // this member's column tile exists (members past the last one only pad)
  unsigned x_off, rs_off;             // byte offsets inside a tile's exchange area
  unsigned row_off, d_off, p_off;     // ... of the thread's values inside 16 rows of [N] floats, a tile's record, a tile's pairs
  unsigned tile_bytes, slot_bytes;

  __device__ __forceinline__ TeamAux(const RingTeamArgs& c, int mem, int at_)
      : map(at_), at(at_), lane(at_ & 63) {
    ct = mem * C16 + map.c;
    j0 = 16 * ct + 4 * map.q + 2 * map.p;
    tile_ok = map.active && ct < 2 * c.KC;
    const unsigned kc = (unsigned)j0 >> 5;
    x_off = kc * CHUNK_BYTES + ((((unsigned)j0 >> 3) & 3) * 16 + map.b) * 16 + (j0 & 7) * 2;
    rs_off = kc * CHUNK_BYTES + 1024 + map.b * 16 + (((unsigned)j0 >> 3) & 3) * 4;
    if (!tile_ok) x_off = NOWHERE;
    // one lane of those that share a row's eight neurons (four lanes of two, or two of four) writes their sum
    if (!tile_ok || ((lane >> 2) & (NPT == 4 ? 1 : 3)) != 0) rs_off = NOWHERE;
    row_off = tile_ok && j0 < c.N ? (unsigned)(map.b * c.N + j0) * 4 : NOWHERE;
    d_off = tile_ok ? (unsigned)(ct * 256 + (map.q * 16 + map.b) * 4 + 2 * map.p) * 2 : NOWHERE;
    // one 16-byte slot per neuron and row quad (see pair_offset; tile = neuron / 16): after the quad transpose a lane has
    // neuron 4q + (lane & 3), both steps (NPT = 4), or neuron 4q + 2p + (lane & 1), step lane & 2 (NPT = 2)
    const int n = NPT == 4 ? 4 * map.q + (lane & 3) : 4 * map.q + 2 * map.p + (lane & 1);
    p_off = tile_ok ? (unsigned)(ct * 1024 + ((map.b >> 2) * 16 + n) * 16 + (NPT == 4 ? 0 : (lane & 2) * 4)) : NOWHERE;
    tile_bytes = (unsigned)c.KC * CHUNK_BYTES;
    slot_bytes = tile_bytes * (unsigned)c.nbt;
  }

  template <int ST>
  __device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t rsrc, unsigned base, const unsigned (&x)[NPT / 2], unsigned r) {
    if constexpr (NPT == 4) {
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{x[0], x[1]}, rsrc, (int)x_off, (int)base, ST);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(x[0], rsrc, (int)x_off, (int)base, ST);
    }
    __builtin_amdgcn_raw_buffer_store_b32(r, rsrc, (int)rs_off, (int)base, ST);
  }
  // publish the thread's NPT values of a tile's state in `slot`
  __device__ __forceinline__ void publish(const RingTeamArgs& c, __amdgpu_buffer_rsrc_t rsrc, int slot, int bt, const float (&v)[NPT]) {
    unsigned x[NPT / 2];
#pragma unroll
    for (int i = 0; i < NPT / 2; ++i) x[i] = not_empty(pack_bf16(v[2 * i], v[2 * i + 1]));
    float s = v[0] + v[1];
    if (c.J0 != 0.f) {
      if constexpr (NPT == 4) {
        const float u = v[2] + v[3];
        s = row_sum8(s, u, dpp_ror<0x12C>(s), dpp_ror<0x12C>(u));    // (row_ror:12: the next four neurons' lane)
      } else {
        s = sum_bits23(s);
      }
    }
    const unsigned r = not_empty(__builtin_bit_cast(unsigned, s));
    const unsigned base = (unsigned)slot * slot_bytes + (unsigned)bt * tile_bytes;
    put<ST_LOCAL>(rsrc, base, x, r);
  }
  __device__ __forceinline__ void refill(const RingTeamArgs& c, __amdgpu_buffer_rsrc_t rsrc, int slot, int bt) {
    unsigned x[NPT / 2];
#pragma unroll
    for (int i = 0; i < NPT / 2; ++i) x[i] = EMPTY;
    const unsigned base = (unsigned)slot * slot_bytes + (unsigned)bt * tile_bytes;
    put<ST_LOCAL>(rsrc, base, x, EMPTY);
  }

  template <int WK>
  __device__ __forceinline__ void sum_shares(const float* share, int buf, float (&v)[NPT]) const {
    const float* src = share + ((size_t)buf * WK * C16 + map.c) * AM::SHARE + map.q * AM::QS + map.b * 4 + 2 * map.p;
    typedef float fN __attribute__((ext_vector_type(NPT)));
    fN a[WK];
#pragma unroll
    for (int w = 0; w < WK; ++w) a[w] = *reinterpret_cast<const fN*>(src + (size_t)w * C16 * AM::SHARE);
    __builtin_amdgcn_sched_barrier(0);            // all reads on their way before the first sum waits
#pragma unroll
    for (int w = 1; w < WK; ++w) a[0] += a[w];
#pragma unroll
    for (int i = 0; i < NPT; ++i) v[i] = a[0][i];
  }

  // NPT floats of the thread's row of an fp32 [B][N] slab, in one load (4-byte alignment is all it needs).  Rows past B
  // read the last row; a quad that reaches past N is read as the row's last NPT neurons, which align() moves into
  // place.  Nothing may touch the values before they are used (a select right behind the load would wait for it), so it
  // is the user who aligns and masks.
  __device__ __forceinline__ void row_load_raw(const float* slab, int N, int B, int bt, float (&v)[NPT]) const {
    const int b = 16 * bt + map.b;
    const float* src = slab + (size_t)(b < B ? b : B - 1) * N + (j0 + NPT <= N ? j0 : N - NPT);
    if constexpr (NPT == 4) {
      const f32x4 a = *reinterpret_cast<const f32x4u*>(src);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = a[i];
    } else {
      const f32x2 a = *reinterpret_cast<const f32x2u*>(src);
      v[0] = a[0];
      v[1] = a[1];
    }
  }
  __device__ __forceinline__ void align(int N, float (&v)[NPT]) const {
    if (N % NPT == 0) return;
    const int sh = j0 + NPT <= N ? 0 : j0 + NPT - N;
    if constexpr (NPT == 4) {
      if (sh & 2) { v[0] = v[2]; v[1] = v[3]; }
      if (sh & 1) { v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; }
    } else {
      if (sh & 1) v[0] = v[1];
    }
  }
  __device__ __forceinline__ void row_load(const float* slab, int N, int B, int bt, float (&v)[NPT]) const {
    row_load_raw(slab, N, B, bt, v);
    align(N, v);
#pragma unroll
    for (int i = 0; i < NPT; ++i) v[i] = (16 * bt + map.b < B && map.active && j0 + i < N) ? v[i] : 0.f;
  }
  // into row block bt of an fp32 [B][N] slab
  __device__ __forceinline__ void row_store(float* slab, int N, int B, int bt, const float (&v)[NPT]) const {
    const int rows = B - 16 * bt < 16 ? B - 16 * bt : 16;
    const __amdgpu_buffer_rsrc_t r = team_buffer(slab + (size_t)16 * bt * N, (size_t)rows * N * 4);
    if (N % NPT == 0) {
      if constexpr (NPT == 4)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{v[0], v[1], v[2], v[3]}), r, (int)row_off, 0, 0);
      else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{v[0], v[1]}), r, (int)row_off, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        const float a = v[i];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, a), r, (int)(j0 + i < N ? row_off + 4 * i : NOWHERE), 0, 0);
      }
    }
  }
  // derivative record: fp16 [t][batch tile][column tile][q][row][4 neurons]
  __device__ __forceinline__ size_t dact_offset(int t, int nbt, int bt, int cts) const {
    return (((size_t)t * nbt + bt) * cts + (ct < cts ? ct : cts - 1)) * 256 + (map.q * 16 + map.b) * 4 + 2 * map.p;
  }
  __device__ __forceinline__ void dact_store(_Float16* base, int t, int nbt, int bt, int cts, const unsigned (&d)[NPT / 2]) const {
    const __amdgpu_buffer_rsrc_t r = team_buffer(base + ((size_t)t * nbt + bt) * cts * 256, base ? (size_t)cts * 512 : 0);
    if constexpr (NPT == 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2{d[0], d[1]}, r, (int)d_off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(d[0], r, (int)d_off, 0, 0);
  }
  // operand copy for the weight gradients: steps 2j (lo) and 2j + 1 (hi) of a neuron's four rows side by side
  __device__ __forceinline__ void pair_put(__bf16* base, int t, int nbt, int bt, int cts, const unsigned (&lo)[NPT / 2],
                                           const unsigned (&hi)[NPT / 2]) const {
    const __amdgpu_buffer_rsrc_t r =
        team_buffer(reinterpret_cast<char*>(base) + ((size_t)(t >> 1) * nbt + bt) * cts * 1024, (size_t)cts * 1024);
    if constexpr (NPT == 4) {
      const u32x2 a = quad_rows4(lo[0], lo[1], lane), d = quad_rows4(hi[0], hi[1], lane);
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{a[0], a[1], d[0], d[1]}, r, (int)p_off, 0, 0);
    } else {
      const u32x2 a = quad_rows2(lo[0], lane), d = quad_rows2(hi[0], lane);
      __builtin_amdgcn_raw_buffer_store_b64((lane & 2) ? d : a, r, (int)p_off, 0, 0);
    }
  }
};

// Gates of one item's 16 rows (a_dim <= 16: one value per auxiliary thread), [k][16] in LDS.
struct TeamGates {
  size_t off;      // of this thread's row and channel in one step of batch tile 0
  int row, lds;
  bool mine;
  __device__ __forceinline__ TeamGates(const RingTeamArgs& c, int at) {
    row = at / c.k;
    const int ch = at - row * c.k;
    mine = row < 16;
    lds = mine ? ch * 16 + row : c.k * 16 * 2;      // (idle threads write to a spare word behind the two buffers)
    off = mine ? (size_t)row * c.T * c.k + ch : 0;
  }
  __device__ __forceinline__ float fetch(const RingTeamArgs& c, int t, int bt) const {
    // (rows past B get some other gate: their operand is zero)
    return c.A[((size_t)16 * bt * c.T + t) * c.k + (16 * bt + row < c.B ? off : 0)];
  }
  __device__ __forceinline__ void put(float* gl, float v) const {
    gl[lds] = v;
  }
};

// The item `ahead` items after (s, j), and its batch tile; clamped to the last one.
struct ItemCursor {
  int s, j;
  __device__ __forceinline__ void advance(int my_nt, int steps) {
    if (j + 1 < my_nt) ++j;
    else if (s + 1 < steps) { j = 0; ++s; }
  }
};

__device__ __forceinline__ bool team_coords(const RingTeamArgs& c, int& team, int& mem) {
  const int y = blockIdx.x >> 3;       // members 8 indices apart: one XCD
  team = (blockIdx.x & 7) + 8 * (y / c.G);
  mem = y % c.G;
  return team < c.nteams;
}

}  // namespace

// Shapes that are built: K chunks per compute wave, column tiles per member, matrices in registers, compute waves, up to how many
// further matrices in LDS there is a kernel for exactly that number, and whether there is one for any number (not where LDS or a cheaper
// shape leaves no call for it).  (kpw * wk chunks cover the contraction; c16 * kpw * mr weight fragments of
// four registers per wave.  Past N = 512 one column tile per member would make teams of more than an XCD's 32 compute
// units; four at 256 < N <= 512 leave LDS room for a further matrix only up to N = 288, where two are as fast: N = 257,
// a_dim 3, B = 1395, T = 60 forward 235 us with four, 233 with two.)
// One to four matrices in LDS with three in registers, or one with nine, are multiplied without a loop, their gates read together and
// no look at whether all of them are silent; us a call of T = 40 with the loop of any number -> without: forward N = 653, 3 channels,
// B = 973 393 -> 358, N = 700, 4 channels, B = 500 239 -> 215, N = 144, 5 channels, B = 900 114 -> 95, N = 300, 9 channels, B = 800
// 291 -> 285; training N = 300, 6 channels, B = 800 500 -> 462; with two of six driven forward 107 -> 109.  One with thirteen: N = 500,
// 13 channels, B = 300 179 -> 184.  One kernel for up to four, each behind a test of the number of channels: N = 653 372, N = 700 222,
// N = 144 101, two of six driven 117.
#define RING_TEAM_SHAPES(X)                                                                                                  \
  X(1, 1, 3, 4, 0, true) X(1, 2, 3, 4, 0, true) X(1, 4, 3, 4, 0, true)                                                       \
  X(1, 1, 3, 8, 3, false) X(1, 2, 3, 8, 4, true) X(1, 4, 3, 8, 3, false) X(1, 1, 9, 8, 1, true) X(1, 2, 13, 8, 0, true)      \
  X(2, 1, 3, 8, 3, false) X(2, 2, 3, 8, 4, true) X(2, 4, 3, 8, 0, false) X(2, 1, 9, 8, 1, true) X(2, 1, 13, 8, 0, true)      \
  X(3, 2, 3, 8, 2, false) X(4, 2, 3, 8, 1, false)

// Launches one team kernel.
template <typename F>
hipError_t ring_team_start(const void* kernel, const RingTeamShape& sh, int G, unsigned lds, hipStream_t st, F&& go) {
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  const RingLaunchGuard::Launch order(ring_launch_guard(), st, G - 1);
  go(dim3((unsigned)sh.grid), dim3(64u * (unsigned)(sh.wk + AUX)), lds);
  return hipGetLastError();
}

