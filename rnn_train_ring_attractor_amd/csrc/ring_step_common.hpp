// Helpers shared by the step-per-launch kernel families (ring_bign.hip, ring_block.hip): run-time-NC layout
// offsets, masked row loads and stores, staging of operand rows and action gates into LDS.
#pragma once
#include "ring_common.hpp"
#include "ring_kernels.hpp"

#include <stdlib.h>
#include <type_traits>

namespace {

constexpr int BN_GATE_KMAX = 64;

// Which (row group, column block) a workgroup takes.  Workgroups go to the eight XCDs round-robin by linear index,
// and every XCD has its own L2.  With the plain (x = row group, y = column block) order each XCD sees every column
// block, i.e. pulls the whole packed weight set out of HBM for itself -- eight fetches of every weight byte per
// step, which is what bounds small batches of wide rings.  When the column blocks divide by eight, XCD x instead
// owns column blocks x * cpx .. (x+1) * cpx - 1 for all row groups: each weight byte leaves HBM once per step and is
// shared through that XCD's L2 by the row groups running side by side.  With fewer than eight column blocks the
// packed weights are small enough for every XCD's L2, and letting several XCDs share a block was measured to cost a
// little, so those grids keep the plain order.  Any placement gives correct results; the mapping only decides what
// the caches see.  xcd_map = 0 keeps the plain order.
__device__ __forceinline__ void step_block_coords(int xcd_map, int& rg, int& cb) {
  const int nrg = gridDim.x, ncb = gridDim.y;
  rg = blockIdx.x;
  cb = blockIdx.y;
  if (xcd_map && (ncb & 7) == 0) {
    const int L = blockIdx.x + nrg * blockIdx.y, xcd = L & 7, w = L >> 3, cpx = ncb >> 3;
    rg = w % nrg;
    cb = xcd * cpx + w / nrg;
  }
}

// RINGATTR_XCD_MAP=0: plain workgroup order (see step_block_coords)
inline int step_xcd_map() {
  const char* v = getenv("RINGATTR_XCD_MAP");
  return (v && v[0] == '0') ? 0 : 1;
}


__device__ __forceinline__ size_t pair_off_rt(int NC, int t, int nbt, int bt, int tile, int lane) {
  return (((((size_t)(t >> 1) * nbt + bt) * (size_t)(4 * NC) + tile) * 64 + lane) * 2 + (t & 1)) * 4;
}

// slot of K position j (neuron), row b in the LDS operand buffer (see write_operand): 16-byte slots, groups padded to XG
__device__ __forceinline__ int op_slot(int j, int b) { return ((j >> 5) * 4 + ((j >> 3) & 3)) * XG + b; }

// fp32 [rows][N] row-major, four consecutive neurons, masked
__device__ __forceinline__ f32x4 load4_masked(const float* slab, int N, int B, int b, int j) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (b >= B || j >= N) return v;
  const float* src = slab + (size_t)b * N + j;
  if ((N & 3) == 0) return *reinterpret_cast<const f32x4*>(src);   // j is a multiple of 4, so j + 3 < N
#pragma unroll
  for (int x = 0; x < 4; ++x)
    if (j + x < N) v[x] = src[x];
  return v;
}

// ---- a workgroup's rows, read in batches of loads that are all on their way together ----
// What a step waited for most was its operand: read four neurons at a time behind a test of row and column, one load
// waited for the one before, sixteen and more of them in a row.  Here rows lie in a buffer that ends with the batch and
// columns past N point past it, so that no load hangs on a branch.  us per step before and after, forward / BPTT:
//   block kernels, 16 channels of which two are driven: N = 1024, B = 64 24.8 -> 14.8 / 38.5 -> 17.4, N = 761, B = 260 24.7 -> 20.0 /
//     56.5 -> 25.2, N = 1000, B = 3000 79 -> 65 / 115 -> 74; all 16 driven, N = 2048, B = 100: 96 -> 76 / 135 -> 80
//   one-tile kernels, 3 channels: N = 600, B = 3000 66.2 -> 64.5 / 85 -> 72, N = 1500, B = 800 70 -> 64 / 81 -> 68

// Rows `first` .. `first + rows - 1` of an array that has `all` of them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* array, size_t first, size_t all, int rows, size_t row_bytes) {
  const size_t left = first < all ? all - first : 0, n = left < (size_t)rows ? left : (size_t)rows;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(array)) + (left ? first * row_bytes : 0), 0,
                                           (int)(n * row_bytes), 0x00020000);
}

constexpr unsigned PAST_ROWS = 0x80000000u;      // (an offset past every buffer: reads zero)

// Neurons j .. j + V - 1 of a buffer's row; those past N are zero.  WHOLE: N is a multiple of four (and j of V = 4).
template <int V, bool WHOLE>
__device__ __forceinline__ f32x4 row_columns(__amdgpu_buffer_rsrc_t r, int row, int N, int j) {
  const unsigned at = (unsigned)(row * N + j) * 4u;
  if constexpr (WHOLE && V == 4) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(j < N ? at : PAST_ROWS), 0, 0));
  } else {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < V; ++x) v[x] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)(j + x < N ? at + 4u * x : PAST_ROWS), 0, 0));
    return v;
  }
}

template <typename F>
__device__ __forceinline__ void with_whole(int N, F&& f) {
  if ((N & 3) == 0) f(std::true_type{});
  else f(std::false_type{});
}

// The state: r_prev as it is.
template <bool WHOLE>
struct StateRows {
  using Raw = f32x4;
  struct Row {};
  static constexpr int BATCH = 8;
  __amdgpu_buffer_rsrc_t r;
  int N;
  __device__ __forceinline__ Row row(int) const { return Row{}; }
  __device__ __forceinline__ Raw load(int row, int j) const { return row_columns<4, WHOLE>(r, row, N, j); }
  __device__ __forceinline__ f32x4 value(const Raw& v, const Row&, int) const { return v; }
};

// BPTT: G = grad_output + carry, g = (alpha F') * G.  LOSS: grad_output is not read but formed from the state history and the
// loss head's row coefficients,  up * (kc cos(phi_j) + ks sin(phi_j) + beta sign(r_j)),  (cos, sin) from the table of
// ring_launch_trig_table.
template <bool LOSS>
struct GradRaw {
  f32x4 v, carry;            // grad_output or the state; carry
  f16x4 d;
};
struct GradTrig { f32x4 t[2]; };
struct GradCoef { float kc, ks, beta; };

template <bool LOSS, bool WHOLE>
struct GradRows {
  struct Raw {
    GradRaw<LOSS> g;
    GradTrig trig;
  };
  using Row = GradCoef;
  static constexpr int BATCH = LOSS ? 4 : 8;
  const RingBpttArgs& p;
  int t, first, NPAD;
  float up;
  bool has_carry;
  __amdgpu_buffer_rsrc_t rows, carry, d;
  // `first`: the workgroup's first row, of `count`; carry and record rows lie in padded [16 * nbt][NPAD] arrays
  __device__ __forceinline__ GradRows(const RingBpttArgs& p_, int t_, int first_, int count, int NPAD_, const float* carry_in, float up_)
      : p(p_), t(t_), first(first_), NPAD(NPAD_), up(up_), has_carry(carry_in != nullptr) {
    const size_t pad = (size_t)16 * p.nbt, f = (size_t)first;
    rows = rows_buffer((LOSS ? p.hist : p.grad_out) + (size_t)t * p.B * p.N, f, (size_t)p.B, count, (size_t)p.N * 4);
    carry = rows_buffer(carry_in, f, has_carry ? pad : f, count, (size_t)NPAD * 4);
    d = rows_buffer(p.dfrag + (size_t)t * pad * NPAD, f, pad, count, (size_t)NPAD * 2);
  }
  __device__ __forceinline__ Row row(int row) const {
    if constexpr (!LOSS) return Row{0.f, 0.f, 0.f};
    const int b = first + row;
    const f32x4 c = p.loss_coef[(size_t)t * p.B + (b < p.B ? b : p.B - 1)];
    const float in = b < p.B ? up : 0.f;
    return Row{b < p.B ? c[0] * in : 0.f, b < p.B ? c[1] * in : 0.f, b < p.B ? c[2] * in : 0.f};
  }
  __device__ __forceinline__ GradRaw<LOSS> load_row(int row, int j) const {
    GradRaw<LOSS> g;
    g.v = row_columns<4, WHOLE>(rows, row, p.N, j);
    g.carry = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(carry, (row * NPAD + j) * 4, 0, 0));
    g.d = __builtin_bit_cast(f16x4, __builtin_amdgcn_raw_buffer_load_b64(d, (row * NPAD + j) * 2, 0, 0));
    return g;
  }
  __device__ __forceinline__ GradTrig load_trig(int j) const {
    GradTrig g;
    if constexpr (LOSS) {
      g.t[0] = *reinterpret_cast<const f32x4*>(p.loss_trig + 2 * j);        // j is a multiple of 4
      g.t[1] = *reinterpret_cast<const f32x4*>(p.loss_trig + 2 * j + 4);
    }
    return g;
  }
  __device__ __forceinline__ Raw load(int row, int j) const { return Raw{load_row(row, j), load_trig(j)}; }
  __device__ __forceinline__ f32x4 value(const Raw& raw, const Row& c, int j) const {
    f32x4 G;
    return form(raw.g, raw.trig, c, j, p.N, has_carry, G);
  }
  static __device__ __forceinline__ f32x4 form(const GradRaw<LOSS>& raw, const GradTrig& trig, const Row& c, int j, int N, bool has_carry, f32x4& G) {
    G = raw.v;
    if constexpr (LOSS) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float r = raw.v[x], cs = trig.t[x >> 1][2 * (x & 1)], sn = trig.t[x >> 1][2 * (x & 1) + 1];
        const float sb = r > 0.f ? c.beta : (r < 0.f ? -c.beta : 0.f);              // beta * sign(r), sign(0) = 0
        G[x] = j + x < N ? fmaf(c.kc, cs, fmaf(c.ks, sn, sb)) : 0.f;
      }
    }
    if (has_carry) G += raw.carry;
    // products rounded on their own (never contracted into the row sum that follows), so that both step-per-launch
    // families form bit-identical g and row sums whatever the compiler does with the surrounding code
    f32x4 g;
    {
#pragma clang fp contract(off)
      g = f32x4{(float)raw.d[0] * G[0], (float)raw.d[1] * G[1], (float)raw.d[2] * G[2], (float)raw.d[3] * G[3]};
    }
    return g;
  }
};

// Stage RT batch tiles' operand rows (bf16, tile i at xb + i * slots) and their fp32 row sums (rs[16 * i + row]).
// Thread (row = tid / 16, sub = tid % 16) walks its row in groups of four neurons, 64 neurons apart (NPAD is a multiple).
template <int RT, typename S>
__device__ __forceinline__ void stage_rows(bf16x8* xb, int slots, float* rs, int NPAD, int tid, const S& src) {
  const int row = tid >> 4, sub = tid & 15;
#pragma unroll 1
  for (int i = 0; i < RT; ++i) {
    float sum = 0.f;
    char* base = reinterpret_cast<char*>(xb + (size_t)i * slots);
    const typename S::Row c = src.row(16 * i + row);
#pragma unroll 1
    for (int g = 0; g < NPAD; g += 64 * S::BATCH) {
      typename S::Raw raw[S::BATCH];
#pragma unroll
      for (int u = 0; u < S::BATCH; ++u) {
        const int at = g + 64 * u;
        raw[u] = src.load(16 * i + row, (at < NPAD ? at : 0) + 4 * sub);       // (past the row: its first again, unused)
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < S::BATCH; ++u) {
        if (g + 64 * u >= NPAD) break;
        const int j = g + 64 * u + 4 * sub;
        const f32x4 v = src.value(raw[u], c, j);
        sum += (v[0] + v[1]) + (v[2] + v[3]);
        const bf16x4 pk = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
        *reinterpret_cast<bf16x4*>(base + (size_t)op_slot(j, row) * 16 + (j & 7) * 2) = pk;
      }
    }
    sum = row16_sum_dpp(sum);
    if (sub == 0) rs[16 * i + row] = sum;
  }
}

__device__ __forceinline__ void store4_masked(float* slab, int N, int B, int b, int j, f32x4 v) {
  if (b >= B || j >= N) return;
  float* dst = slab + (size_t)b * N + j;
  if ((N & 3) == 0) {
    *reinterpret_cast<f32x4*>(dst) = v;
    return;
  }
#pragma unroll
  for (int x = 0; x < 4; ++x)
    if (j + x < N) dst[x] = v[x];
}

// V consecutive neurons (V in {1, 2, 4}) of one batch row as a zero-padded f32x4
template <int V>
__device__ __forceinline__ f32x4 loadv_masked(const float* slab, int N, int B, int b, int j) {
  if constexpr (V == 4) return load4_masked(slab, N, B, b, j);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (b >= B) return v;
  const float* src = slab + (size_t)b * N + j;
#pragma unroll
  for (int x = 0; x < V; ++x)
    if (j + x < N) v[x] = src[x];
  return v;
}

template <int V>
__device__ __forceinline__ void storev_masked(float* slab, int N, int B, int b, int j, f32x4 v) {
  if constexpr (V == 4) {
    store4_masked(slab, N, B, b, j, v);
    return;
  }
  if (b >= B) return;
  float* dst = slab + (size_t)b * N + j;
#pragma unroll
  for (int x = 0; x < V; ++x)
    if (j + x < N) dst[x] = v[x];
}

__device__ __forceinline__ void stage_gates(float* gl, const float* __restrict__ A, int k, int T, int B, int t, int bt, int tid) {
  for (int idx = tid; idx < 16 * k; idx += 256) {
    const int row = idx / k, c = idx - row * k, b = 16 * bt + row;
    gl[row * BN_GATE_KMAX + c] = b < B ? A[((size_t)b * T + t) * k + c] : 0.f;
  }
}

// bit c set <=> channel c has a non-zero gate in some of the 16 rows (same value in every lane)
__device__ __forceinline__ unsigned long long active_channels(const float* gl, int k, int lane) {
  unsigned long long m = 0;
  for (int c0 = 0; c0 < k; c0 += 4) {
    const int c = c0 + (lane >> 4);
    const bool nz = c < k && gl[(lane & 15) * BN_GATE_KMAX + c] != 0.f;
    const unsigned long long bal = __ballot(nz);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if ((bal >> (16 * j)) & 0xffffull) m |= 1ull << (c0 + j);
  }
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)m), hi = __builtin_amdgcn_readfirstlane((unsigned)(m >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

}  // namespace
