// Teams of one: forward and BPTT for 17 <= N <= 128, a workgroup per RW batch rows, all weights in registers.
//
// Up to N = 128 and six channels a wave per column tile holds the rows of [Wo | Wa] for its 16 neurons in registers for the
// whole sequence, and the state goes from step to step through LDS: one workgroup barrier a step, no hand-over through L2, no
// gathering, no second launch.  Every sum is a row's own, in the same order whatever the batch and RW.
//
// A step of a wave: the whole state as MFMA operands from LDS (KCT fragments), the products of 1 + a_dim matrices (weights
// are the A operand, so a lane ends up with four consecutive neurons of one batch row and a gate is one scalar per lane),
// activation or g, the new operand back to LDS.  What goes to HBM is issued behind the barrier, under the next operand's
// way out of LDS; what comes from there is fetched two steps ahead.  Every store is a buffer store that drops what a lane or
// a step has nothing to store for: without branches the compiler knows how many memory operations follow a load and waits
// for that load alone.
//
// What bounds a step is one compute unit's vector issue: with 16 rows a lane's four activations are most of some 130
// instructions, four cycles each, on two waves a SIMD (0.87 us a step, gelu, N = 120).  While compute units are idle a workgroup
// takes RW = 4 or 8 rows instead (0.54 and 0.69 us): columns RW .. 15 of the products repeat the first ones, and each of the
// lanes that hold a row works on its own one or two of the four neurons.  What is left then is the chain of a step: operand
// out of LDS, 24 products on each matrix pipe (390 of some 1300 cycles), activation, operand into LDS.
// us per step, N = 120, two channels, forward / BPTT, against teams of eight workgroups: B = 64 0.54 / 0.65 (0.76 / 0.95),
// B = 1024 0.57 / 0.95 (forward 1.12), B = 4096 0.90 / 1.27 (forward 1.44; 3.1 TB/s in the BPTT).
//
// The order of the sums is that of a team with one compute wave (chunks one after the other, row sums in groups of eight
// neurons), so ring_team_rebuild_kernel gives the same record with wk = 1.
#include "ring_team.hpp"

namespace {

constexpr int ONE_MATS[] = {3, 7};      // matrices in registers: the smallest that holds 1 + a_dim

// What a lane has: EPL consecutive neurons from j0 on of row `row` of the workgroup's RW, in everything that is stored.
template <int RW>
struct OneLane {
  static constexpr int EPL = RW / 4;
  int lane, q, row, sub, j0, at_row;    // at_row: the row's place in the whole batch, clamped into it
  bool live;                            // the row is in the batch
  unsigned row_off, d_off, p_off;       // byte offsets in the workgroup's [RW][N] block, a tile's record, a tile's pairs
  __device__ __forceinline__ OneLane(int w, int lane_, int first, int N, int B) : lane(lane_), q(lane_ >> 4) {
    const int n = lane & 15;
    row = n % RW;
    sub = n / RW;
    j0 = 16 * w + 4 * q + sub * EPL;
    live = first + row < B;
    at_row = live ? first + row : B - 1;
    row_off = j0 < N && live ? (unsigned)(row * N + j0) * 4 : NOWHERE;
    const int r16 = first % 16 + row;
    d_off = (unsigned)(w * 256 + (q * 16 + r16) * 4 + sub * EPL) * 2;
    const int slot = w * 1024 + ((r16 >> 2) * 16 + 4 * q) * 16;
    if constexpr (RW == 16) p_off = (unsigned)(slot + (lane & 3) * 16);
    else if constexpr (RW == 8) p_off = (unsigned)(slot + (2 * sub + (lane & 1)) * 16 + (lane & 2) * 4);
    else p_off = (unsigned)(slot + sub * 16 + (lane & 3) * 4);
  }
  // the lane's place in an operand (bytes) and its row sum's
  __device__ __forceinline__ int x_at() const { return ((j0 >> 3) * RW + row) * 16 + (j0 & 7) * 2; }
  __device__ __forceinline__ int rs_at() const { return (j0 >> 3) * RW + row; }

  // V values of the lane's row of an fp32 [B][N] slab from neuron j on, which is a multiple of V; a group that reaches past N
  // is read as the row's last V values, which align() moves into place
  template <int V>
  __device__ __forceinline__ void row_load(const float* slab, int N, int j, float (&v)[V]) const {
    typedef float fV __attribute__((ext_vector_type(V), aligned(4)));
    const fV a = *reinterpret_cast<const fV*>(slab + ((size_t)at_row * N + (j + V <= N ? j : N - V)));
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = a[i];
  }
  __device__ __forceinline__ void row_load(const float* slab, int N, int j, float (&v)[1]) const {
    v[0] = slab[(size_t)at_row * N + (j < N ? j : N - 1)];
  }
  template <int V>
  __device__ __forceinline__ void align(int N, int j, float (&v)[V]) const {
    if constexpr (V == 1) return;
    if (N % V == 0) return;
    const int sh = j + V <= N ? 0 : j + V - N;
    if constexpr (V == 4) {
      if (sh & 2) { v[0] = v[2]; v[1] = v[3]; }
      if (sh & 1) { v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; }
    } else if constexpr (V == 2) {
      if (sh & 1) v[0] = v[1];
    }
  }
  // into the workgroup's rows of a [B][N] slab
  __device__ __forceinline__ void row_store(__amdgpu_buffer_rsrc_t r, int N, const float (&v)[EPL]) const {
    if (N % EPL == 0) {
      if constexpr (EPL == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{v[0], v[1], v[2], v[3]}), r, (int)row_off, 0, 0);
      else if constexpr (EPL == 2) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{v[0], v[1]}), r, (int)row_off, 0, 0);
      else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v[0]), r, (int)row_off, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < EPL; ++i) {
        const float a = v[i];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, a), r, (int)(j0 + i < N ? row_off + 4 * i : NOWHERE), 0, 0);
      }
    }
  }
  // the operand copy for the weight gradients: steps 2j (lo) and 2j + 1 (hi) of a neuron's four rows side by side
  __device__ __forceinline__ void pair_store(__amdgpu_buffer_rsrc_t r, const float (&lo)[EPL], const float (&hi)[EPL]) const {
    if constexpr (EPL == 4) {
      const u32x2 a = quad_rows4(pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), lane), d = quad_rows4(pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3]), lane);
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{a[0], a[1], d[0], d[1]}, r, (int)p_off, 0, 0);
    } else if constexpr (EPL == 2) {
      const u32x2 a = quad_rows2(pack_bf16(lo[0], lo[1]), lane), d = quad_rows2(pack_bf16(hi[0], hi[1]), lane);
      __builtin_amdgcn_raw_buffer_store_b64((lane & 2) ? d : a, r, (int)p_off, 0, 0);
    } else {                            // (a quad has a neuron's four rows: lane 0 writes rows 0 and 1 of lo, 1 the others, 2 and 3 hi's)
      const int both = (int)pack_bf16(lo[0], hi[0]);
      const unsigned a = (unsigned)__builtin_amdgcn_update_dpp(0, both, 0x88, 0xF, 0xF, false);      // quad_perm [0,2,0,2]
      const unsigned d = (unsigned)__builtin_amdgcn_update_dpp(0, both, 0xDD, 0xF, 0xF, false);      // quad_perm [1,3,1,3]
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_amdgcn_perm(d, a, (lane & 2) ? 0x07060302u : 0x05040100u), r, (int)p_off, 0, 0);
    }
  }
  // the lane's own of a product's four neurons
  __device__ __forceinline__ void own(const f32x4& p, float (&v)[EPL]) const {
    if constexpr (EPL == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = p[i];
    } else if constexpr (EPL == 2) {
      v[0] = sub ? p[2] : p[0];
      v[1] = sub ? p[3] : p[1];
    } else {
      const float lo = (sub & 1) ? p[1] : p[0], hi = (sub & 1) ? p[3] : p[2];
      v[0] = (sub & 2) ? hi : lo;
    }
  }
};

template <int KCT, int MR, int RW>
struct OneLds {
  bf16x8 x[2][KCT * 4 * RW];         // operand: [chunk][q][row] x 8 neurons
  float rs[2][KCT * 4 * RW];         // fp32 sums of the unrounded values, groups of eight neurons (zeros without a J0 term)
  float gates[2][(MR - 1) * RW + 1]; // [channel][row], and a word for idle threads
};

// The lane's values into an operand, with their row sum.
template <int KCT, int MR, int RW>
__device__ __forceinline__ void one_put(OneLds<KCT, MR, RW>& L, int buf, const OneLane<RW>& o, bool sums, const float (&v)[RW / 4]) {
  char* const x = reinterpret_cast<char*>(L.x[buf]) + o.x_at();
  float s, u;                        // sums of neurons 4q, 4q + 1 and of 4q + 2, 4q + 3, in the lanes of sub 0
  if constexpr (RW == 16) {
    *reinterpret_cast<u32x2*>(x) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    s = v[0] + v[1];
    u = v[2] + v[3];
  } else if constexpr (RW == 8) {
    *reinterpret_cast<unsigned*>(x) = pack_bf16(v[0], v[1]);
    s = v[0] + v[1];
    u = dpp_ror<0x128>(s);                                 // row_ror:8
  } else {
    const float next = dpp_ror<0x12C>(v[0]);               // row_ror:12, the lane four further on
    const unsigned two = pack_bf16(v[0], next);
    if ((o.sub & 1) == 0) *reinterpret_cast<unsigned*>(x) = two;
    s = v[0] + next;
    u = dpp_ror<0x128>(s);
  }
  if (sums) {
    const unsigned si = __builtin_bit_cast(unsigned, s), ui = __builtin_bit_cast(unsigned, u);
    const auto a = __builtin_amdgcn_permlane16_swap(si, si, false, false), d = __builtin_amdgcn_permlane16_swap(ui, ui, false, false);
    const unsigned s0 = a[0], s2 = a[1], s1 = d[0], s3 = d[1];        // (of the even and of the odd lane row)
    const float sum = row_sum8(__builtin_bit_cast(float, s0), __builtin_bit_cast(float, s1), __builtin_bit_cast(float, s2), __builtin_bit_cast(float, s3));
    if ((o.q & 1) == 0 && o.sub == 0) L.rs[buf][o.rs_at()] = sum;
  }
}

// The wave's weight fragments: output neurons of its column tile, all chunks; matrices past a_dim are zero.
// The workgroup takes in the whole ring, which a short call feels.  Rows off 16-byte boundaries come in 16-byte loads too,
// where a chunk is whole, and nothing is loaded for matrices that are not there.  us a call, T = 20, three channels, teams of
// eight workgroups, here a word at a time with seven matrices, so: N = 101, B = 64: 27 39 22, B = 20000: 164 232 151; N = 65,
// B = 1: 26.6 29.4 21.2; five channels, N = 127, B = 64: 33 44 30.
// What is left is instruction issue, so few are spent on a value: a chunk's mask is made once for all matrices and put on pairs,
// addresses are 32-bit offsets, and rows of the transposed matrix that are not there are past a buffer's end.  us of a training
// pass, teams of eight, a mask and an address a value, so: N = 65, B = 1, T = 1, six channels 37.2 43.7 37.9; N = 128, B = 64, T = 3,
// six 40.4 43.1 39.5; N = 101, B = 300, T = 8, six 81.7 80.2 75.3; forward, N = 65, B = 300, T = 8, four 16.6 17.3 16.0.  The
// forward of one to three steps stays up to 1.3 us behind the teams (N = 101, four channels: 9.3 and 10.5), 4.7 where rows are
// off their boundaries and all seven matrices there (N = 127, six: 13.2 and 17.9; a row of 128 bytes touches two lines twice).
template <int KCT, int MR, bool TR>
__device__ __forceinline__ void one_weights(const RingTeamArgs& c, int w, int lane, bf16x8 (&wt)[MR][KCT]) {
  const int q = lane >> 4, out = 16 * w + (lane & 15);
  const unsigned o = out < c.N ? out : c.N - 1;
  u32x4 keep[KCT];                     // what of a fragment is in the matrix
#pragma unroll
  for (int kc = 0; kc < KCT; ++kc)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int left = out < c.N ? c.N - (32 * kc + 8 * q + 2 * i) : 0;
      keep[kc][i] = left > 1 ? 0xFFFFFFFFu : (left > 0 ? 0xFFFFu : 0u);
    }
  auto load = [&](auto how) {
    constexpr int HOW = decltype(how)::value, F = MR * KCT, BATCH = 4;
    const unsigned row = (unsigned)c.N * 4u, at = HOW == WEIGHT_COLUMNS ? 8 * q * row + 4u * o : o * row + 32u * q;      // bytes
    auto fetch = [&](WeightLoad& l, int m, int kc) {
      const float* W = m == 0 || m > c.k ? c.Wo : c.Wa + (size_t)(m - 1) * c.N * c.N;
      if constexpr (HOW == WEIGHT_COLUMNS) {           // (rows past the matrix are past the buffer: zeros)
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(W), 0, (int)(c.N * row), 0x00020000);
#pragma unroll
        for (int x = 0; x < 8; ++x)
          l.v[x] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)(at + (32 * kc + x) * row), 0, 0));
      } else if (HOW == WEIGHT_ROWS && 32 * kc + 32 <= c.N) {
        const char* src = reinterpret_cast<const char*>(W + 32 * kc) + at;
        const f32x4 lo = *reinterpret_cast<const f32x4u*>(src), hi = *reinterpret_cast<const f32x4u*>(src + 16);
#pragma unroll
        for (int x = 0; x < 4; ++x) { l.v[x] = lo[x]; l.v[4 + x] = hi[x]; }
      } else if (HOW == WEIGHT_ROWS) {
        const unsigned last = c.N - 1, k0 = 32 * kc + 8 * q;
        const char* src = reinterpret_cast<const char*>(W);
#pragma unroll
        for (int x = 0; x < 8; ++x) l.v[x] = *reinterpret_cast<const float*>(src + (o * row + 4u * (k0 + x < last ? k0 + x : last)));
      } else {
        weight_load<HOW>(l, W, c.N, out, 32 * kc + 8 * q);
      }
    };
#pragma unroll
    for (int f0 = 0; f0 < F; f0 += BATCH) {
      if (f0 / KCT > c.k) {
#pragma unroll
        for (int f = f0; f < f0 + BATCH && f < F; ++f) wt[f / KCT][f % KCT] = bf16x8{};
        continue;
      }
      WeightLoad l[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (f0 + i < F) fetch(l[i], (f0 + i) / KCT, (f0 + i) % KCT);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const int m = (f0 + i) / KCT, kc = (f0 + i) % KCT;
        if (f0 + i < F) {
          u32x4 f;
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            f[x] = pack_bf16(l[i].v[2 * x], l[i].v[2 * x + 1]) & keep[kc][x];
            if (f0 % KCT != 0 || BATCH > KCT) f[x] = m <= c.k ? f[x] : 0u;      // (otherwise the batch is one matrix)
          }
          asm volatile("" : "+v"(f));              // (here, not at its first use: twice the registers until then)
          wt[m][kc] = __builtin_bit_cast(bf16x8, f);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (TR) load(std::integral_constant<int, WEIGHT_COLUMNS>{});
  else if ((c.N & 3) == 0) load(std::integral_constant<int, WEIGHT_ROWS4>{});
  else load(std::integral_constant<int, WEIGHT_ROWS>{});
}

// J1 P_0 + J0 rowsum + sum_m gate_m P_m for the lane's four neurons.  `between` runs while the operand is on its way out of
// LDS, dot(m, P_m) with every channel's products.
template <int KCT, int MR, int RW, typename Between, typename Dot>
__device__ __forceinline__ f32x4 one_products(const RingTeamArgs& c, const OneLds<KCT, MR, RW>& L, int buf, const bf16x8 (&wt)[MR][KCT],
                                              const OneLane<RW>& o, Between&& between, Dot&& dot) {
  constexpr int GROUP = 4;                                 // chains of products at a time
  bf16x8 x[KCT];
  float rs[KCT], g[MR];
#pragma unroll
  for (int kc = 0; kc < KCT; ++kc) x[kc] = L.x[buf][(kc * 4 + o.q) * RW + o.row];
#pragma unroll
  for (int kc = 0; kc < KCT; ++kc) rs[kc] = L.rs[buf][(kc * 4 + o.q) * RW + o.row];
#pragma unroll
  for (int m = 1; m < MR; ++m) g[m] = L.gates[buf][(m - 1) * RW + o.row];
  __builtin_amdgcn_sched_barrier(0);
  between();
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc;
#pragma unroll
  for (int m0 = 0; m0 < MR; m0 += GROUP) {
    if (m0 > c.k) break;                                   // (channels past a_dim in a started group: zero weights and gates)
    f32x4 P[GROUP];
#pragma unroll
    for (int m = 0; m < GROUP; ++m) P[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KCT; ++kc)
#pragma unroll
      for (int m = 0; m < GROUP; ++m)
        if (m0 + m < MR) P[m] = mfma16(wt[m0 + m < MR ? m0 + m : 0][kc], x[kc], P[m]);
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      if (m0 + m == 0) {
        float sum = 0.f;
#pragma unroll
        for (int kc = 0; kc < KCT; ++kc) sum += rs[kc];
        const float j0r = c.J0 * sum_bits45(sum);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(c.J1, P[0][i], j0r);
      } else if (m0 + m < MR) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(g[m0 + m < MR ? m0 + m : 0], P[m][i], acc[i]);
        dot(m0 + m, P[m]);
      }
    }
  }
  return acc;
}

// Gates of a step's rows: a value per thread.
template <int RW>
struct OneGates {
  unsigned at;
  int lds;
  bool mine;
  __device__ __forceinline__ OneGates(const RingTeamArgs& c, int first, int tid, int spare) {
    const int ch = tid / RW, row = tid % RW;
    mine = ch < c.k && first + row < c.B;
    lds = tid < spare ? tid : spare;
    at = mine ? (unsigned)(row * c.T * c.k + ch) : 0u;
  }
  __device__ __forceinline__ const float* rows(const RingTeamArgs& c, int first) const { return c.A + (size_t)(first < c.B ? first : 0) * c.T * c.k; }
  __device__ __forceinline__ float fetch(const float* step) const { return step[at]; }
  __device__ __forceinline__ void put(float* dst, float v) const { dst[lds] = mine ? v : 0.f; }
};

// A buffer that starts `step` bytes further on every time it is asked for: what a time step stores, without multiplications.
struct OneStream {
  char* base;
  size_t step;
  unsigned bytes;
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t next() {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)bytes, 0x00020000);
    base += step;
    return r;
  }
};

// Without a J0 term no step writes row sums: zeros once, because J0 times what LDS was left with need not be zero.
template <int KCT, int MR, int RW>
__device__ __forceinline__ void one_no_sums(OneLds<KCT, MR, RW>& L, int tid) {
  for (int i = tid; i < 2 * KCT * 4 * RW; i += 128 * KCT) (&L.rs[0][0])[i] = 0.f;
}

__device__ __forceinline__ int one_rows(int first, int B, int RW) { return B - first < 0 ? 0 : (B - first < RW ? B - first : RW); }

}  // namespace

// ------------------------------------------------------------------------------------------------
// Forward.  p.dfrag / p.rfrag may be null together (inference).
// ------------------------------------------------------------------------------------------------
template <int KCT, int MR, int RW, int ACT>
__global__ __launch_bounds__(128 * KCT, 2) void ring_team_one_fwd_kernel(RingFwdArgs p, RingTeamArgs c) {
  __shared__ OneLds<KCT, MR, RW> L;
  constexpr int EPL = RW / 4;
  typedef _Float16 fE __attribute__((ext_vector_type(EPL)));
  const int tid = threadIdx.x, first = blockIdx.x * RW, bt = first / 16, N = p.N, B = p.B, T = p.T;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), rows = one_rows(first, B, RW);
  const OneLane<RW> o(w, tid & 63, first, N, B);
  const OneGates<RW> og(c, first, tid, (MR - 1) * RW);
  const float* gate_at = og.rows(c, first);
  int left = T;                        // steps whose gates have not been asked for
  auto gate_next = [&] {
    const float g = og.fetch(gate_at);
    gate_at += --left > 0 ? c.k : 0;
    return g;
  };
  const float g0 = gate_next();
  float gA = gate_next(), gB = gate_next();
  bf16x8 wt[MR][KCT];
  one_weights<KCT, MR, false>(c, w, tid & 63, wt);
  const float oma = 1.f - p.alpha;
  const ActScale asc = act_scale_make(p.alpha);
  const bool sums = c.J0 != 0.f;
  float r[EPL], before[EPL];
  fE d;
  o.row_load(p.r_init, N, o.j0, r);
  o.align(N, o.j0, r);
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    r[i] = o.live && o.j0 + i < N ? r[i] : 0.f;
    before[i] = 0.f;
    d[i] = (_Float16)0.f;
  }
  if (!sums) one_no_sums(L, tid);
  one_put(L, 0, o, sums, r);
  og.put(L.gates[0], g0);
  const size_t tile_d = (size_t)c.cts * 256, tile_p = (size_t)c.cts * 512;
  OneStream to_hist{reinterpret_cast<char*>(p.hist + (size_t)first * N), (size_t)B * N * 4, (unsigned)(rows * N * 4)};
  OneStream to_d{reinterpret_cast<char*>(p.dfrag + (size_t)bt * tile_d), p.nbt * tile_d * 2, p.dfrag ? (unsigned)tile_d * 2 : 0u};
  OneStream to_p{reinterpret_cast<char*>(p.rfrag + (size_t)bt * tile_p), p.nbt * tile_p * 2, p.rfrag ? (unsigned)tile_p * 2 : 0u};
  // what a step left in r, d and before
  auto store = [&](bool even, bool last) {
    o.row_store(to_hist.next(), N, r);
    const __amdgpu_buffer_rsrc_t rd = to_d.next();
    if constexpr (EPL == 4) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, d), rd, (int)o.d_off, 0, 0);
    else if constexpr (EPL == 2) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, d), rd, (int)o.d_off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, d), rd, (int)o.d_off, 0, 0);
    if (even) {                        // before: the state the step began with; r: what the next one begins with
      float hi[EPL];
#pragma unroll
      for (int i = 0; i < EPL; ++i) hi[i] = last ? 0.f : r[i];
      o.pair_store(to_p.next(), before, hi);
    }
  };
  lds_barrier();
  auto step = [&](int t, bool even, float& g) {
    og.put(L.gates[even ? 1 : 0], g);                      // the next step's, fetched two steps ago
    const f32x4 all = one_products(c, L, even ? 0 : 1, wt, o, [&] {
      g = gate_next();
      if (t > 0) store(!even, false);
    }, [](int, const f32x4&) {});
    float pre[EPL];
    o.own(all, pre);
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      ActRecord<ACT> rd;
      const float aF = rd.apply(pre[i], asc);
      before[i] = r[i];
      r[i] = o.j0 + i < N ? fmaf(oma, r[i], aF) : 0.f;       // (rows past B stay zero by themselves)
      d[i] = rd.once(asc);
    }
    one_put(L, even ? 1 : 0, o, sums, r);
    lds_barrier();
  };
  step(0, true, gA);
  int t = 1;
  for (; t + 1 < T; t += 2) {
    step(t, false, gB);
    step(t + 1, true, gA);
  }
  if (t < T) step(t, false, gB);
  store((T & 1) != 0, true);
}

// ------------------------------------------------------------------------------------------------
// BPTT, reverse time; g of step t is the operand of round T - 1 - t.
// ------------------------------------------------------------------------------------------------
template <int KCT, int MR, int RW, bool GA>
__global__ __launch_bounds__(128 * KCT, 2) void ring_team_one_bptt_kernel(RingBpttArgs p, RingTeamArgs c) {
  __shared__ OneLds<KCT, MR, RW> L;
  __shared__ float ga[GA ? 2 : 1][GA ? (MR - 1) * 2 * KCT * RW : 1];        // dL/dA shares [channel][wave][row]
  constexpr int EPL = RW / 4;
  typedef _Float16 fE __attribute__((ext_vector_type(EPL)));
  const int tid = threadIdx.x, first = blockIdx.x * RW, bt = first / 16, N = p.N, B = p.B, T = p.T;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), rows = one_rows(first, B, RW);
  const OneLane<RW> o(w, tid & 63, first, N, B);
  const OneGates<RW> og(c, first, tid, (MR - 1) * RW);
  const float oma = 1.f - p.alpha;
  const bool sums = c.J0 != 0.f, loss = p.loss_coef != nullptr;
  const size_t tile_d = (size_t)c.cts * 256, tile_p = (size_t)c.cts * 512;
  const float* const grads = loss ? p.hist : p.grad_out;
  const char* const coef = loss ? reinterpret_cast<const char*>(p.loss_coef + o.at_row) : reinterpret_cast<const char*>(c.Wo);
  const int jq = 16 * w + 4 * o.q;     // the product's four neurons
  struct In {                          // of step t; gate: of step t - 1
    float go[EPL];
    fE d;
    f32x3 cf;
    float rp[GA ? 4 : 1];
    float gate;
  };
  // (past the first step everything stays where it is: what is fetched there is not used)
  int left = T;                        // steps that have not been asked for
  const float *gate_at = og.rows(c, first) + (size_t)(T - 1) * c.k, *grad_at = grads + (size_t)(T - 1) * B * N;
  const float* prev_at = T > 1 ? p.hist + (size_t)(T - 2) * B * N : p.r_init;
  const char *d_at = reinterpret_cast<const char*>(p.dfrag + ((size_t)(T - 1) * p.nbt + bt) * tile_d), *coef_at = coef + (loss ? (size_t)(T - 1) * B * 16 : 0);
  auto fetch = [&](In& in) {
    gate_at -= left > 1 ? c.k : 0;
    in.gate = og.fetch(gate_at);
    o.row_load(grad_at, N, o.j0, in.go);
    in.d = *reinterpret_cast<const fE*>(d_at + o.d_off);
    in.cf = *reinterpret_cast<const f32x3*>(coef_at);      // (without the loss head: unused)
    if constexpr (GA) o.row_load(prev_at, N, jq, in.rp);
    if (--left > 0) {
      grad_at -= (size_t)B * N;
      d_at -= p.nbt * tile_d * 2;
      coef_at -= loss ? (size_t)B * 16 : 0;
      prev_at = left > 1 ? prev_at - (size_t)B * N : p.r_init;
    }
  };
  In inA, inB;
  og.put(L.gates[0], og.fetch(gate_at));
  if (!sums) one_no_sums(L, tid);
  bf16x8 wt[MR][KCT];
  one_weights<KCT, MR, true>(c, w, tid & 63, wt);
  fetch(inA);
  fetch(inB);
  float cs[EPL], sn[EPL], up = 0.f;
#pragma unroll
  for (int i = 0; i < EPL; ++i) { cs[i] = 0.f; sn[i] = 0.f; }
  if (loss) {
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const float phi = 6.2831853071795864769f * (float)(o.j0 + i) / (float)N;
      cs[i] = cosf(phi);
      sn[i] = sinf(phi);
    }
    up = (p.loss_upstream ? p.loss_upstream[0] : 1.f) * p.loss_inv_rows;
  }
  // dL/dA of round s (step T - 1 - s): the waves' shares in wave order; what a thread or a round has not goes nowhere
  auto flush = [&](int s) {
    if constexpr (GA) {
      const int ch = tid / RW, row = tid % RW;
      const float* src = ga[s & 1] + (ch < MR - 1 ? ch : 0) * 2 * KCT * RW + row;
      float v = 0.f;
#pragma unroll
      for (int x = 0; x < 2 * KCT; ++x) v += src[x * RW];
      const bool mine = og.mine && s >= 0;
      const __amdgpu_buffer_rsrc_t r = team_buffer(p.grad_A + (size_t)first * T * c.k, (size_t)rows * T * c.k * 4);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)(mine ? (unsigned)((row * T + T - 1 - s) * c.k + ch) * 4 : NOWHERE), 0, 0);
    }
  };
  char* g_at = reinterpret_cast<char*>(p.gfrag + ((size_t)((T - 1) >> 1) * p.nbt + bt) * tile_p);
  float carry[EPL], gg[EPL], held[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) carry[i] = gg[i] = held[i] = 0.f;
  const bool last_round = p.grad_r_init || GA;             // whether the first step's products are wanted
  auto round = [&](int s, bool one, In& in) {              // one: the first of the unrolled loop's two
    const int t = T - 1 - s, buf = one ? 0 : 1;
    float G[EPL], rp[4] = {0.f, 0.f, 0.f, 0.f};
    o.align(N, o.j0, in.go);
    const float kc = in.cf[0] * up, ks = in.cf[1] * up, beta = in.cf[2] * up;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      float go = in.go[i];
      if (loss) {
        const float r = go;
        go = fmaf(kc, cs[i], fmaf(ks, sn[i], r > 0.f ? beta : (r < 0.f ? -beta : 0.f)));
      }
      const bool ok = o.live && o.j0 + i < N;
      G[i] = ok ? go + carry[i] : 0.f;
      held[i] = gg[i];
      gg[i] = ok ? (float)in.d[i] * G[i] : 0.f;       // the record carries alpha
    }
    if constexpr (GA) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rp[i] = in.rp[i];
      o.align(N, jq, rp);
#pragma unroll
      for (int i = 0; i < 4; ++i) rp[i] = o.live && jq + i < N ? rp[i] : 0.f;
    }
    one_put(L, buf, o, sums, gg);
    const float gate = in.gate;
    auto out = [&] {
      fetch(in);
      // an even step's, with the step behind it (held: zero before the first round)
      o.pair_store(team_buffer(g_at, (t & 1) ? 0 : tile_p * 2), gg, held);
      g_at -= (t & 1) ? 0 : p.nbt * tile_p * 2;
      flush(s - 1);
    };
    if (t == 0 && !last_round) {
      out();
      return;
    }
    lds_barrier();
    og.put(L.gates[buf ^ 1], gate);
    float dots[GA ? MR : 1];
    const f32x4 all = one_products(c, L, buf, wt, o, out, [&](int m, const f32x4& P) {
      if constexpr (GA) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) v = fmaf(P[i], rp[i], v);
        dots[m] = v;
      }
    });
    float acc[EPL];
    o.own(all, acc);
#pragma unroll
    for (int i = 0; i < EPL; ++i) carry[i] = fmaf(oma, G[i], acc[i]);
    if constexpr (GA) {
#pragma unroll
      for (int m = 1; m < MR; ++m) {
        const float v = sum_bits45(dots[m]);
        if (m <= c.k && (tid & 63) < RW) ga[buf][((m - 1) * 2 * KCT + w) * RW + (tid & 63)] = v;
      }
    }
  };
  for (int s = 0; s < T; s += 2) {
    round(s, true, inA);
    if (s + 1 < T) round(s + 1, false, inB);
  }
  if constexpr (GA) {
    lds_barrier();
    flush(T - 1);
  }
  if (p.grad_r_init) o.row_store(team_buffer(p.grad_r_init + (size_t)first * N, (size_t)rows * N * 4), N, carry);
}

// Widths and channels that the registers hold, at any batch.  Forward, T = 20, eleven widths from 17 to 128, as a share of the
// time on teams of eight and, at large batches, on the streaming kernels, one / two / four / six channels: B = 64
// 0.77-0.83 / 0.78-0.82 / 0.72-0.98 / 0.59-0.91, B = 2000 0.52-0.81 / 0.53-0.82 / 0.49-0.77 / 0.39-0.64, B = 8192 0.43-0.62 / 0.44-0.64 /
// 0.33-0.62 / 0.25-0.49, B = 20000 0.34-0.54 / 0.31-0.57 / 0.32-0.98 / 0.24-0.83.  Training at B = 20000 0.33-0.84.
bool ring_team_one_applicable(int N, int k) { return N >= 17 && N <= 128 && k >= 1 && k < ONE_MATS[1]; }

namespace {

// Rows per workgroup: as few as the compute units can take one workgroup each (B = 1024: 4 rows 0.59 us a step, 8 rows 0.69,
// 16 rows 0.87; B = 4096: 2.42, 1.35, 0.90).
int one_rows_per_group(int nbt) {
  return nbt <= 64 ? 4 : (nbt <= 128 ? 8 : 16);
}

template <int KCT, int MR, int RW>
hipError_t one_fwd(const RingFwdArgs& a, const RingTeamArgs& c, hipStream_t st) {
  const dim3 grid((unsigned)(a.nbt * (16 / RW))), block(128 * KCT);
  switch (a.act) {
    case ACT_RELU: RING_LAUNCH((ring_team_one_fwd_kernel<KCT, MR, RW, ACT_RELU>), grid, block, 0, st, a, c); break;
    case ACT_GELU: RING_LAUNCH((ring_team_one_fwd_kernel<KCT, MR, RW, ACT_GELU>), grid, block, 0, st, a, c); break;
    case ACT_TANH: RING_LAUNCH((ring_team_one_fwd_kernel<KCT, MR, RW, ACT_TANH>), grid, block, 0, st, a, c); break;
    case ACT_SILU: RING_LAUNCH((ring_team_one_fwd_kernel<KCT, MR, RW, ACT_SILU>), grid, block, 0, st, a, c); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int KCT, int MR, int RW>
hipError_t one_bptt(const RingBpttArgs& a, const RingTeamArgs& c, hipStream_t st) {
  const dim3 grid((unsigned)(a.nbt * (16 / RW))), block(128 * KCT);
  if (a.grad_A) RING_LAUNCH((ring_team_one_bptt_kernel<KCT, MR, RW, true>), grid, block, 0, st, a, c);
  else RING_LAUNCH((ring_team_one_bptt_kernel<KCT, MR, RW, false>), grid, block, 0, st, a, c);
  return hipGetLastError();
}

template <typename F>
hipError_t one_shape(int N, int k, int nbt, F&& go) {
  const int rw = one_rows_per_group(nbt);
  const auto rows = [&](auto kct, auto mr) {
    if (rw == 4) return go(kct, mr, std::integral_constant<int, 4>{});
    if (rw == 8) return go(kct, mr, std::integral_constant<int, 8>{});
    return go(kct, mr, std::integral_constant<int, 16>{});
  };
  const auto mats = [&](auto kct) {
    if (k < ONE_MATS[0]) return rows(kct, std::integral_constant<int, ONE_MATS[0]>{});
    return rows(kct, std::integral_constant<int, ONE_MATS[1]>{});
  };
  return N <= 64 ? mats(std::integral_constant<int, 2>{}) : mats(std::integral_constant<int, 4>{});
}

}  // namespace

hipError_t ring_launch_team_one_fwd(const RingFwdArgs& a, const RingTeamArgs& c, hipStream_t st) {
  if (!ring_team_one_applicable(a.N, a.k) || c.cts != (a.N <= 64 ? 4 : 8) || !a.hist || (a.dfrag != nullptr) != (a.rfrag != nullptr))
    return hipErrorInvalidValue;
  return one_shape(a.N, a.k, a.nbt, [&](auto kct, auto mr, auto rw) { return one_fwd<decltype(kct)::value, decltype(mr)::value, decltype(rw)::value>(a, c, st); });
}

hipError_t ring_launch_team_one_bptt(const RingBpttArgs& a, const RingTeamArgs& c, hipStream_t st) {
  if (!ring_team_one_applicable(a.N, a.k) || c.cts != (a.N <= 64 ? 4 : 8)) return hipErrorInvalidValue;
  return one_shape(a.N, a.k, a.nbt, [&](auto kct, auto mr, auto rw) { return one_bptt<decltype(kct)::value, decltype(mr)::value, decltype(rw)::value>(a, c, st); });
}
