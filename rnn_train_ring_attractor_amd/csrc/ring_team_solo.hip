// The team kernels' arithmetic (ring_team.hpp) by single workgroups, which need no other workgroup to be resident.
//
// ring_team_rebuild_kernel makes the saved record out of a given state history: every (step, batch tile) stands alone, so
// nothing is handed over.
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
          float aF, aD;
          act_scaled<ACT>(tot[cc][r][i], asc, aF, aD);
          d[i] = (_Float16)aD;
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
