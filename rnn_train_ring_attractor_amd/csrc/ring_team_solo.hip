// The team kernels' arithmetic (ring_team.hpp) by single workgroups, which need no other workgroup to be resident.
//
// ring_team_rebuild_kernel makes the saved record out of a given state history: every (step, batch tile) stands alone, so
// nothing is handed over.  ring_team_solo_fwd_kernel and ring_team_solo_bptt_kernel run the time loops of the teams whose
// members did not become resident together.
//
// The order of every sum is that of the team kernels (K chunks by compute wave, matrices one after the other, the waves'
// shares in wave order), so the bits are the same.
#include "ring_team.hpp"

namespace {

// One step's operand in LDS: [K chunk][64 lanes] x 16 bytes, lane (q, row) with neurons 32 kc + 8 q .. + 7, and the sum of
// each such group of eight.
struct SoloOperand {
  bf16x8* x;
  float* rs;
};

// Eight neurons of one row: the lane's operand and their sum.
__device__ __forceinline__ void solo_put(const SoloOperand& o, int at, const float (&v)[8]) {
  u32x4 x;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = not_empty(pack_bf16(v[2 * i], v[2 * i + 1]));
  o.x[at] = __builtin_bit_cast(bf16x8, x);
  o.rs[at] = row_sum8(v[0] + v[1], v[2] + v[3], v[4] + v[5], v[6] + v[7]);
}

// Eight consecutive values of a row of an fp32 [B][N] slab from neuron j on; zero past the row's or the batch's end.
__device__ __forceinline__ void solo_row8(const float* __restrict__ slab, int N, int B, int b, int j, float (&v)[8]) {
  if (b < B && j + 8 <= N) {
    const f32x4 lo = *reinterpret_cast<const f32x4u*>(slab + (size_t)b * N + j);
    const f32x4 hi = *reinterpret_cast<const f32x4u*>(slab + (size_t)b * N + j + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = lo[i]; v[4 + i] = hi[i]; }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = b < B && j + i < N ? slab[(size_t)b * N + j + i] : 0.f;
  }
}

}  // namespace

// ------------------------------------------------------------------------------------------------
// Rebuild of the record (alpha F' and the bf16 operand copy) from bump_history.  R / 2 batch tiles x 2 steps per workgroup
// share every weight fragment, which comes packed in bf16 (natural tile order): at R = 4 a fragment's load (1 KiB through
// a compute unit that takes in some 64 B per clock) and its four products on one of four matrix pipes take equally long.
// ------------------------------------------------------------------------------------------------
// A wave takes two column tiles at a time and keeps the items' operands of one compute wave's chunks in registers for all
// matrices (read from LDS per matrix they would take twice what LDS delivers); the next matrix's fragments travel during
// the products.  us, gelu, against the recurrence run again by the team forward: N = 360, a_dim 3, B = 100, T = 75: 50
// (117); N = 120, B = 64, T = 120: 11 (99); N = 512, B = 2048, T = 60: 347 (303); N = 1024, B = 2048, T = 60: 1155 (1075).
// KPW: K chunks of one compute wave of a team (wk of them).
template <int R, int KPW, int ACT>
__global__ __launch_bounds__(512) void ring_team_rebuild_kernel(RingFwdArgs p, RingTeamArgs c, int wk) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int KC = c.KC, XC = wk * KPW, tid = threadIdx.x, nthreads = blockDim.x, nw = nthreads >> 6;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4, b = lane & 15, T = p.T, k = c.k;
  // (the waves' chunks past the last one hold zeros)
  bf16x8* const x = reinterpret_cast<bf16x8*>(lds);                        // [R][XC][64]
  float* const rs = reinterpret_cast<float*>(x + (size_t)R * XC * 64);     // [R][XC][64]
  float* const gates = rs + (size_t)R * XC * 64;                           // [R][k][16]
  // item r: batch tile bt0 + r / 2, step t0 + r % 2
  const int groups = (p.nbt + R / 2 - 1) / (R / 2), bt0 = (int)(blockIdx.x % groups) * (R / 2), t0 = 2 * (int)(blockIdx.x / groups);
  auto tile = [&](int r) { return bt0 + r / 2; };
  auto there = [&](int r) { return tile(r) < p.nbt && t0 + (r & 1) < T; };

  for (int u = tid; u < R * XC * 64; u += nthreads) {
    const int r = u / (XC * 64), at = u - r * XC * 64, l = at & 63, t = t0 + (r & 1);
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.f;
    if (there(r))
      solo_row8(t == 0 ? p.r_init : p.hist + (size_t)(t - 1) * p.B * p.N, p.N, p.B, 16 * tile(r) + (l & 15),
                32 * (at >> 6) + 8 * (l >> 4), v);
    solo_put(SoloOperand{x + (size_t)r * XC * 64, rs + (size_t)r * XC * 64}, at, v);
  }
  for (int u = tid; u < R * k * 16; u += nthreads) {
    const int r = u / (k * 16), ch = u / 16 % k, row = 16 * tile(r) + (u & 15);
    gates[u] = there(r) && row < p.B ? c.A[((size_t)row * T + t0 + (r & 1)) * k + ch] : 0.f;
  }
  lds_barrier();

  // the operand copy: steps t0 and t0 + 1 of a neuron's four rows side by side
  for (int u = tid; u < R * KC * 64; u += nthreads) {
    const int h = u / (2 * KC * 64), ct = u / 64 % (2 * KC), rq = u >> 4 & 3, n = u & 15, j = 16 * ct + n;
    const int bt = bt0 + h;
    if (bt >= p.nbt) break;
    const __bf16* lo = reinterpret_cast<const __bf16*>(x + (size_t)2 * h * XC * 64 + (j >> 5) * 64 + ((j >> 3) & 3) * 16 + 4 * rq) + (j & 7);
    const __bf16* hi = lo + (size_t)XC * 64 * 8;
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[i] = lo[i * 8]; o[4 + i] = hi[i * 8]; }
    *reinterpret_cast<bf16x8*>(p.rfrag + ((((size_t)(t0 >> 1) * p.nbt + bt) * c.cts + ct) * 64 + (u & 63)) * 8) = o;
  }

  unsigned driven = 0;                           // channels with a gate that is not zero (zero-padded signals: two of many)
  for (int m = 1; m <= k; ++m) {
    bool any = false;
#pragma unroll
    for (int r = 0; r < R; ++r) any |= gates[((size_t)r * k + m - 1) * 16 + b] != 0.f;
    driven |= __ballot(any) ? 1u << m : 0u;
  }
  driven = __builtin_amdgcn_readfirstlane(driven);

  const ActScale asc = act_scale_make(p.alpha);
  const bf16x8* const W = reinterpret_cast<const bf16x8*>(p.Wpack) + lane;         // [1 + k][cts][cts / 2][64]
  const int shares = wk < KC ? wk : KC;                                          // compute waves of a team with a chunk
  bf16x8 f[2][KPW], next[2][KPW];
  auto fetch = [&](int pair, int cw, int m) {    // one matrix's fragments of column tiles 2 pair, 2 pair + 1 and wave cw's chunks
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk)
        next[cc][kk] = W[(((size_t)m * c.cts + 2 * pair + cc) * (c.cts / 2) + cw + wk * kk) * 64];
  };
  if (w < KC) fetch(w, 0, 0);
  for (int pair = w; pair < KC; pair += nw) {
    f32x4 tot[2][R], acc[2][R], P[2][R];
    for (int cw = 0; cw < shares; ++cw) {
      bf16x8 xv[R][KPW];
      float sum[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        sum[r] = 0.f;
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk) {
          const size_t at = ((size_t)r * XC + cw + wk * kk) * 64 + lane;
          xv[r][kk] = x[at];
          sum[r] += rs[at];
        }
      }
      // P = this matrix's products; the next one's fragments are fetched meanwhile
      auto products = [&](unsigned left) {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int kk = 0; kk < KPW; ++kk) f[cc][kk] = next[cc][kk];
        const bool wrap = cw + 1 == shares, last = pair + nw >= KC;        // (the very last fetch repeats itself, unused)
        fetch(left == 0 && wrap && !last ? pair + nw : pair, left != 0 ? cw : (wrap ? 0 : cw + 1), left != 0 ? __builtin_ctz(left) : 0);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int r = 0; r < R; ++r) P[cc][r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk)
#pragma unroll
          for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < R; ++r) P[cc][r] = mfma16(f[cc][kk], xv[r][kk], P[cc][r]);
      };
      products(driven);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float j0r = c.J0 * sum_bits45(sum[r]);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[cc][r][i] = fmaf(c.J1, P[cc][r][i], j0r);
      }
      for (unsigned left = driven; left;) {
        const int m = __builtin_ctz(left);
        left &= left - 1;
        products(left);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float g = gates[((size_t)r * k + m - 1) * 16 + b];
#pragma unroll
          for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[cc][r][i] = fmaf(g, P[cc][r][i], acc[cc][r][i]);
        }
      }
#pragma unroll
      for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int r = 0; r < R; ++r) tot[cc][r] = cw == 0 ? acc[cc][r] : tot[cc][r] + acc[cc][r];
    }
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (!there(r)) continue;
        f16x4 d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ActRecord<ACT> rd;
          rd.apply(tot[cc][r][i], asc);
          d[i] = rd.once(asc);
        }
        *reinterpret_cast<f16x4*>(p.dfrag + ((((size_t)t0 + (r & 1)) * p.nbt + tile(r)) * c.cts + 2 * pair + cc) * 256 + (q * 16 + b) * 4) = d;
      }
  }
}

template <int R, int KPW>
static hipError_t launch_rebuild(const RingFwdArgs& a, const RingTeamArgs& c, int wk, hipStream_t st) {
  const size_t lds = (size_t)R * (wk * KPW * 1280 + c.k * 64);
  const size_t blocks = (size_t)((a.nbt + R / 2 - 1) / (R / 2)) * ((a.T + 1) / 2);
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const int rounds = (c.KC + 7) / 8, waves = (c.KC + rounds - 1) / rounds;     // (all waves work in every round)
  auto go = [&](auto kern) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    RING_LAUNCH(kern, dim3((unsigned)blocks), dim3(64 * waves), lds, st, a, c, wk);
    return hipGetLastError();
  };
  switch (a.act) {
    case ACT_RELU: return go(ring_team_rebuild_kernel<R, KPW, ACT_RELU>);
    case ACT_GELU: return go(ring_team_rebuild_kernel<R, KPW, ACT_GELU>);
    case ACT_TANH: return go(ring_team_rebuild_kernel<R, KPW, ACT_TANH>);
    case ACT_SILU: return go(ring_team_rebuild_kernel<R, KPW, ACT_SILU>);
    default: return hipErrorInvalidValue;
  }
}

// Two tiles per workgroup up to N = 512 (past that the registers and LDS do not hold four items' operands), where that
// leaves every compute unit something to do.
hipError_t ring_launch_team_rebuild(const RingFwdArgs& a, const RingTeamArgs& c, int wk, hipStream_t st) {
  if (!a.dfrag || !a.rfrag || !a.hist || !a.Wpack) return hipErrorInvalidValue;
  const bool four = c.KC <= 16 && (long)((a.nbt + 1) / 2) * ((a.T + 1) / 2) >= 512;
  switch ((c.KC + wk - 1) / wk) {
    case 1: return four ? launch_rebuild<4, 1>(a, c, wk, st) : launch_rebuild<2, 1>(a, c, wk, st);
    case 2: return four ? launch_rebuild<4, 2>(a, c, wk, st) : launch_rebuild<2, 2>(a, c, wk, st);
    case 3: return launch_rebuild<2, 3>(a, c, wk, st);
    case 4: return launch_rebuild<2, 4>(a, c, wk, st);
    default: return hipErrorInvalidValue;
  }
}

// ------------------------------------------------------------------------------------------------
// Forward and BPTT of the teams that did not gather, a workgroup per batch tile that goes through the team's members one
// after the other.  The weights are read in fp32 from memory every step: tens of times slower than a team, and hardly
// ever needed.  Workgroups of gathered teams leave at once: the launch and the wait for the members cost a call 3 to 4 us
// (N = 256, B = 1, T = 100: 127 -> 130; N = 120, B = 64, T = 120 in teams of eight, forward and backward: 238 -> 242).
// ------------------------------------------------------------------------------------------------
namespace {

constexpr int SOLO_WAVES = 8, SOLO_C16 = 4;

struct SoloLds {       // byte offsets into dynamic LDS
  unsigned x, rs, state, gates, ga, trig, total;
};
__host__ __device__ inline SoloLds solo_lds(int KC, int k, bool ga, bool trig) {
  SoloLds l;
  unsigned at = 0;
  l.x = at;
  at += 2u * KC * 1024;                          // two operands, this step's and the next one's
  l.rs = at;
  at += 2u * KC * 256;
  l.state = at;
  at += 2u * KC * 1024;                          // [column tile][64 lanes] x 4 neurons: the state, or (1 - alpha) G
  l.gates = at;
  at += (unsigned)k * 64;
  l.ga = at;
  at += ga ? SOLO_WAVES * (unsigned)k * 64 * 2 : 0;       // (weight-resident order: two column tiles' shares)
  l.trig = at;
  at += trig ? (unsigned)KC * 256 : 0;           // (cos, sin) of every neuron's angle
  l.total = at;
  return l;
}

__device__ __forceinline__ bool solo_needed(const RingTeamArgs& c, int bt) {
  const unsigned long long v = *team_word(c, bt % c.nteams);      // (written by the launch in front)
  for (int x = 0; x < 8; ++x)
    if (team_complete(v, c.G, x)) return false;
  return true;
}

template <bool TR>
__device__ __forceinline__ bf16x8 solo_weight(const RingTeamArgs& c, int m, int ct, int kc, int lane) {
  const int out = 16 * ct + (lane & 15), k0 = 32 * kc + 8 * (lane >> 4);
  const float* W = m == 0 ? c.Wo : c.Wa + (size_t)(m - 1) * c.N * c.N;
  WeightLoad l;
  if constexpr (TR) weight_load<WEIGHT_COLUMNS>(l, W, c.N, out, k0);
  else if ((c.N & 3) == 0) weight_load<WEIGHT_ROWS4>(l, W, c.N, out, k0);
  else weight_load<WEIGHT_ROWS>(l, W, c.N, out, k0);
  return weight_fragment(l, c.N, out, k0, m == 0 ? c.scale0 : 1.f, m == 0 ? c.shift0 : 0.f);
}

// What member `mem` of the team adds up for its column tiles: tot[cc], lane (q, row) with neurons 4q .. 4q + 3 of tile
// mem * c16 + cc.  GA: also the member's dL/dA shares, from r_prev in rp, into ga[k][16].
// Weight-resident order (c.rows): the ungated sum starts from `start` (the BPTT's (1 - alpha) G), and a share of dL/dA is a
// column tile's: ga[cc][k][16].
template <bool TR, bool GA>
__device__ __forceinline__ void solo_products(const RingTeamArgs& c, const SoloOperand& o, const float* gates,
                                              const f32x4 (&rp)[SOLO_C16], const f32x4* start, float* ga, int mem, int lane,
                                              f32x4 (&tot)[SOLO_C16]) {
  const int b = lane & 15;
  for (int cw = 0; cw < c.wk && cw < c.KC; ++cw) {
    f32x4 acc[SOLO_C16];
    float sum = 0.f;
    auto chunks = [&](auto&& use) {              // the wave's K chunks in its order
      for (int i = 0; i < (c.rows ? 8 : c.KC); i += c.wk) {
        const int kc = c.rows && !TR ? rows_chunk(i) : cw + i;
        if (kc < c.KC) use(kc);
      }
    };
    chunks([&](int kc) { sum += o.rs[kc * 64 + lane]; });
    const float j0r = c.J0 * sum_bits45(sum);
    for (int m = 0; m <= c.k; ++m) {
      const float g = m == 0 ? 0.f : gates[(m - 1) * 16 + b];
      if (!GA && m >= c.mr && __ballot(g != 0.f) == 0) continue;
      float d = 0.f;
#pragma unroll
      for (int cc = 0; cc < SOLO_C16; ++cc) {
        if (cc >= c.c16) continue;
        f32x4 P = {0.f, 0.f, 0.f, 0.f};
        if (TR && c.rows && m == 0 && mem * c.c16 + cc < 2 * c.KC) P = start[(mem * c.c16 + cc) * 64];
        chunks([&](int kc) { P = mfma16(solo_weight<TR>(c, m, mem * c.c16 + cc, kc, lane), o.x[kc * 64 + lane], P); });
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[cc][i] = m == 0 ? fmaf(c.J1, P[i], j0r) : fmaf(g, P[i], acc[cc][i]);
          if (GA) d = fmaf(P[i], rp[cc][i], d);
        }
        if (GA && m > 0 && c.rows) {
          d = sum_bits45(d);
          if (lane < 16) ga[(cc * c.k + m - 1) * 16 + b] = d;
          d = 0.f;
        }
      }
      if (GA && m > 0 && !c.rows) {
        d = sum_bits45(d);
        if (lane < 16) ga[(m - 1) * 16 + b] = (cw == 0 ? 0.f : ga[(m - 1) * 16 + b]) + d;
      }
    }
#pragma unroll
    for (int cc = 0; cc < SOLO_C16; ++cc)
      if (cc < c.c16) tot[cc] = cw == 0 ? acc[cc] : tot[cc] + acc[cc];
  }
}

// Four neurons of a row from neuron j on; zero past the row's or the batch's end.
__device__ __forceinline__ f32x4 solo_row4(const float* __restrict__ slab, int N, int B, int b, int j) {
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = b < B && j + i < N ? slab[(size_t)b * N + j + i] : 0.f;
  return v;
}
__device__ __forceinline__ void solo_row4_store(float* __restrict__ slab, int N, int B, int b, int j, const f32x4& v) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (b < B && j + i < N) slab[(size_t)b * N + j + i] = v[i];
}

// The lane's four neurons of column tile ct into the operand (all lanes of the wave).
__device__ __forceinline__ void solo_put4(const SoloOperand& o, int ct, int lane, const f32x4& v) {
  const int q = lane >> 4, b = lane & 15, j = 16 * ct + 4 * q, at = (j >> 5) * 64 + ((j >> 3) & 3) * 16 + b;
  const u32x2 x = {not_empty(pack_bf16(v[0], v[1])), not_empty(pack_bf16(v[2], v[3]))};
  *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(o.x + at) + (j & 7) * 2) = x;
  const float s = v[0] + v[1], u = v[2] + v[3], s2 = __shfl_xor(s, 16), u2 = __shfl_xor(u, 16);
  if (!(q & 1)) o.rs[at] = row_sum8(s, u, s2, u2);
}

// A pair of steps of the copy for the weight gradients (hi null: zeros).
// (split: in the weight-resident kernels' tile order, neuron j in column j % 64 / 4 of tile 4 (j / 64) + j % 4)
__device__ __forceinline__ void solo_pair(__bf16* base, int t, int nbt, int bt, int cts, int KC, int tid, const bf16x8* lo, const bf16x8* hi, bool split) {
  for (int u = tid; u < 2 * KC * 64; u += 64 * SOLO_WAVES) {
    const int ct = u >> 6, rq = u >> 4 & 3, j = 16 * ct + (u & 15);
    const size_t at = ((size_t)(j >> 5) * 64 + ((j >> 3) & 3) * 16 + 4 * rq) * 8 + (j & 7);
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = reinterpret_cast<const __bf16*>(lo)[at + i * 8];
      o[4 + i] = hi ? reinterpret_cast<const __bf16*>(hi)[at + i * 8] : (__bf16)0.f;
    }
    const int slot = split ? (4 * (j >> 6) + (j & 3)) * 64 + rq * 16 + ((j & 63) >> 2) : ct * 64 + (u & 63);
    *reinterpret_cast<bf16x8*>(base + (((size_t)(t >> 1) * nbt + bt) * cts * 64 + slot) * 8) = o;
  }
}

// The lane's four values of the derivative record (neurons 16 ct + 4q .., row lane & 15), in either order.
__device__ __forceinline__ size_t solo_dact_at(const RingTeamArgs& c, int t, int nbt, int bt, int ct, int lane, int i) {
  const size_t tile = ((size_t)t * nbt + bt) * c.cts * 256;
  if (!c.rows) return tile + ct * 256 + lane * 4 + i;
  const int j = 16 * ct + 4 * (lane >> 4) + i, b = lane & 15;
  return tile + ((j >> 6) * 64 + (b >> 2) * 16 + ((j & 63) >> 2)) * 16 + (j & 3) * 4 + (b & 3);
}

__device__ __forceinline__ void solo_gates(const RingTeamArgs& c, float* gates, int t, int bt, int tid) {
  for (int u = tid; u < c.k * 16; u += 64 * SOLO_WAVES) {
    const int row = 16 * bt + (u & 15);
    gates[u] = row < c.B ? c.A[((size_t)row * c.T + t) * c.k + (u >> 4)] : 0.f;
  }
}

}  // namespace

template <int ACT>
__global__ __launch_bounds__(64 * SOLO_WAVES) void ring_team_solo_fwd_kernel(RingFwdArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int bt = blockIdx.x;
  if (!solo_needed(c, bt)) return;
  const int KC = c.KC, N = p.N, B = p.B, T = p.T, tid = threadIdx.x, lane = tid & 63, q = lane >> 4, b = 16 * bt + (lane & 15);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SoloLds L = solo_lds(KC, c.k, false, false);
  auto operand = [&](int i) {
    return SoloOperand{reinterpret_cast<bf16x8*>(lds + L.x) + (size_t)i * KC * 64, reinterpret_cast<float*>(lds + L.rs) + (size_t)i * KC * 64};
  };
  f32x4* const state = reinterpret_cast<f32x4*>(lds + L.state) + lane;
  float* const gates = reinterpret_cast<float*>(lds + L.gates);
  const float oma = 1.f - p.alpha;
  const ActScale asc = act_scale_make(p.alpha);

  for (int ct = w; ct < 2 * KC; ct += SOLO_WAVES) {
    const f32x4 r = solo_row4(p.r_init, N, B, b, 16 * ct + 4 * q);
    state[ct * 64] = r;
    solo_put4(operand(0), ct, lane, r);
  }
  for (int t = 0; t < T; ++t) {
    const SoloOperand cur = operand(t & 1), next = operand((t + 1) & 1);
    solo_gates(c, gates, t, bt, tid);
    lds_barrier();
    for (int mem = w; mem < c.G; mem += SOLO_WAVES) {
      f32x4 x[SOLO_C16];
      const f32x4 none[SOLO_C16] = {};
      solo_products<false, false>(c, cur, gates, none, nullptr, nullptr, mem, lane, x);
#pragma unroll
      for (int cc = 0; cc < SOLO_C16; ++cc) {
        const int ct = mem * c.c16 + cc, j = 16 * ct + 4 * q;
        if (cc >= c.c16 || ct >= 2 * KC) continue;
        const f32x4 r = state[ct * 64];
        f32x4 rn;
        f16x4 d;
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          float aF[2];
          const float x2[2] = {x[cc][i], x[cc][i + 1]};
          ActRecord<ACT> rd[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) aF[h] = rd[h].apply(x2[h], asc);
          const f16x2 both = __builtin_bit_cast(f16x2, ActRecord<ACT>::pair(asc, rd[0], rd[1], !c.rows || (c.rows == 2 && (j & 32) && t + 1 < T)));
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            rn[i + h] = j + i + h < N ? fmaf(oma, r[i + h], aF[h]) : 0.f;
            d[i + h] = !c.rows || (b < B && j + i + h < N) ? both[h] : (_Float16)0.f;
          }
        }
        state[ct * 64] = rn;
        solo_put4(next, ct, lane, rn);
        solo_row4_store(p.hist + (size_t)t * B * N, N, B, b, j, rn);
        if (p.dfrag) {
          if (c.rows) {
#pragma unroll
            for (int i = 0; i < 4; ++i) p.dfrag[solo_dact_at(c, t, p.nbt, bt, ct, lane, i)] = d[i];
          } else {
            *reinterpret_cast<f16x4*>(p.dfrag + solo_dact_at(c, t, p.nbt, bt, ct, lane, 0)) = d;
          }
        }
      }
    }
    lds_barrier();
    if (p.rfrag && (t & 1) == 0) solo_pair(p.rfrag, t, p.nbt, bt, c.cts, KC, tid, cur.x, t + 1 < T ? next.x : nullptr, c.rows != 0);
  }
}

template <bool GA>
__global__ __launch_bounds__(64 * SOLO_WAVES) void ring_team_solo_bptt_kernel(RingBpttArgs p, RingTeamArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int bt = blockIdx.x;
  if (!solo_needed(c, bt)) return;
  const int KC = c.KC, N = p.N, B = p.B, T = p.T, k = c.k, tid = threadIdx.x, lane = tid & 63, q = lane >> 4, b = 16 * bt + (lane & 15);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool loss = p.loss_coef != nullptr;
  const SoloLds L = solo_lds(KC, k, GA, loss);
  auto operand = [&](int i) {
    return SoloOperand{reinterpret_cast<bf16x8*>(lds + L.x) + (size_t)i * KC * 64, reinterpret_cast<float*>(lds + L.rs) + (size_t)i * KC * 64};
  };
  f32x4* const state = reinterpret_cast<f32x4*>(lds + L.state) + lane;
  float* const gates = reinterpret_cast<float*>(lds + L.gates);
  float* const ga = reinterpret_cast<float*>(lds + L.ga) + (size_t)w * k * 32;
  f32x2* const trig = reinterpret_cast<f32x2*>(lds + L.trig);
  const float oma = 1.f - p.alpha;
  float up = 0.f;
  if (loss) {
    for (int j = tid; j < 32 * KC; j += 64 * SOLO_WAVES) {
      const float phi = 6.2831853071795864769f * (float)j / (float)N;
      trig[j] = f32x2{cosf(phi), sinf(phi)};
    }
    up = (p.loss_upstream ? p.loss_upstream[0] : 1.f) * p.loss_inv_rows;
    lds_barrier();
  }

  // g of step t from what is carried into it, into an operand; keeps (1 - alpha) G
  auto form_g = [&](int t, int ct, const f32x4& carry, const SoloOperand& o) {
    const int j = 16 * ct + 4 * q;
    const f32x4 in = solo_row4((loss ? p.hist : p.grad_out) + (size_t)t * B * N, N, B, b, j);
    f16x4 d;
    if (c.rows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = p.dfrag[solo_dact_at(c, t, p.nbt, bt, ct, lane, i)];
    } else {
      d = *reinterpret_cast<const f16x4*>(p.dfrag + solo_dact_at(c, t, p.nbt, bt, ct, lane, 0));
    }
    float kc = 0.f, ks = 0.f, beta = 0.f;
    if (loss && b < B) {
      const ring_f32x4 cf = p.loss_coef[(size_t)t * B + b];
      kc = cf[0] * up;
      ks = cf[1] * up;
      beta = cf[2] * up;
    }
    f32x4 gg, keep;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float go = in[i];
      if (loss) {
        const float r = go;
        const f32x2 a = trig[j + i];
        go = fmaf(kc, a[0], fmaf(ks, a[1], r > 0.f ? beta : (r < 0.f ? -beta : 0.f)));
      }
      const bool ok = b < B && j + i < N;
      const float G = ok ? go + carry[i] : 0.f;
      gg[i] = ok ? (float)d[i] * G : 0.f;
      keep[i] = oma * G;
    }
    state[ct * 64] = keep;
    solo_put4(o, ct, lane, gg);
  };

  for (int ct = w; ct < 2 * KC; ct += SOLO_WAVES) form_g(T - 1, ct, f32x4{0.f, 0.f, 0.f, 0.f}, operand(0));
  lds_barrier();
  if (((T - 1) & 1) == 0) solo_pair(p.gfrag, T - 1, p.nbt, bt, c.cts, KC, tid, operand(0).x, nullptr, c.rows != 0);
  const int steps = (p.grad_r_init || GA) ? T : T - 1;
  for (int s = 0; s < steps; ++s) {
    const SoloOperand cur = operand(s & 1), next = operand((s + 1) & 1);
    const int t = T - 1 - s;                     // the products' step
    solo_gates(c, gates, t, bt, tid);
    lds_barrier();
    for (int mem = w; mem < c.G; mem += SOLO_WAVES) {
      f32x4 x[SOLO_C16], rp[SOLO_C16] = {};
      if constexpr (GA) {
#pragma unroll
        for (int cc = 0; cc < SOLO_C16; ++cc)
          if (cc < c.c16) {
            rp[cc] = solo_row4(t == 0 ? p.r_init : p.hist + (size_t)(t - 1) * B * N, N, B, b, 16 * (mem * c.c16 + cc) + 4 * q);
            if (c.rows) {
#pragma unroll
              for (int i = 0; i < 4; ++i) rp[cc][i] = (float)(__bf16)rp[cc][i];
            }
          }
      }
      solo_products<true, GA>(c, cur, gates, rp, state, ga, mem, lane, x);
      if constexpr (GA) {
        const int parts = c.rows ? c.c16 : 1;
        if (lane < 16 && b < B)
          for (int u = 0; u < parts * k; ++u) c.ga_part[(((size_t)(mem * parts + u / k) * T + t) * k + u % k) * B + b] = ga[u * 16 + lane];
      }
#pragma unroll
      for (int cc = 0; cc < SOLO_C16; ++cc) {
        const int ct = mem * c.c16 + cc;
        if (cc >= c.c16 || ct >= 2 * KC) continue;
        const f32x4 carry = c.rows ? x[cc] : state[ct * 64] + x[cc];
        if (t > 0) form_g(t - 1, ct, carry, next);
        else if (p.grad_r_init) solo_row4_store(p.grad_r_init, N, B, b, 16 * ct + 4 * q, carry);
      }
    }
    lds_barrier();
    if (t > 0 && ((t - 1) & 1) == 0) solo_pair(p.gfrag, t - 1, p.nbt, bt, c.cts, KC, tid, next.x, cur.x, c.rows != 0);
  }
}

// (launched past RING_LAUNCH: the slot's kernel is the team kernel in front)
template <typename K, typename Args>
static hipError_t launch_solo(K kern, const Args& a, const RingTeamArgs& c, unsigned lds, hipStream_t st) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)c.nbt), dim3(64 * SOLO_WAVES), lds, st, a, c);
  return hipGetLastError();
}

hipError_t ring_launch_team_solo_fwd(const RingFwdArgs& a, const RingTeamArgs& c, hipStream_t st) {
  const unsigned lds = solo_lds(c.KC, c.k, false, false).total;
  switch (a.act) {
    case ACT_RELU: return launch_solo(ring_team_solo_fwd_kernel<ACT_RELU>, a, c, lds, st);
    case ACT_GELU: return launch_solo(ring_team_solo_fwd_kernel<ACT_GELU>, a, c, lds, st);
    case ACT_TANH: return launch_solo(ring_team_solo_fwd_kernel<ACT_TANH>, a, c, lds, st);
    case ACT_SILU: return launch_solo(ring_team_solo_fwd_kernel<ACT_SILU>, a, c, lds, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t ring_launch_team_solo_bptt(const RingBpttArgs& a, const RingTeamArgs& c, hipStream_t st) {
  const unsigned lds = solo_lds(c.KC, c.k, a.grad_A != nullptr, a.loss_coef != nullptr).total;
  return a.grad_A ? launch_solo(ring_team_solo_bptt_kernel<true>, a, c, lds, st) : launch_solo(ring_team_solo_bptt_kernel<false>, a, c, lds, st);
}
