// One launch per time step for wide rings, forward without a saved record ("panel" kernels).
//
// What bounds a step here is how often the weights travel from the caches into the compute units: at N = 2048 with 16
// channels they are 143 MB, far more than the L2s hold, and ring_block.hip pulls every fragment into eight compute
// units (32 rows x 64 neurons each): 1.1 GB per step at B = 256.  A workgroup here takes a panel of up to 128 rows x 16
// neurons and ALL (1 + a_dim) matrices of it at once: a fragment is fetched by B / 128 workgroups and feeds eight MFMAs,
// and the operand rows, which no longer fit LDS as a whole, stream through it in stages of four K chunks.
//   * A (matrix, column tile) pair is a virtual column; the four waves share out a workgroup's virtual columns in
//     contiguous runs of at most five.  A wave holds the products of its run with every row tile (up to 160
//     accumulators), so weight fragments go straight from global memory to the one wave that needs them (eight chunks
//     ahead), and operand fragments are read from LDS once per wave.
//   * Per K chunk a workgroup with R row tiles and V virtual columns loads (R + V) KiB for R * V MFMAs: 8 + 17 KiB
//     against 544 matrix-pipe cycles at B = 256 and 16 channels.  What is left is the rate at which a compute unit takes
//     in lines that miss its L2; see panel_shape.
//   * The operand arrives as bf16 MFMA fragments: one launch converts the initial state, every step's epilogue the state it
//     makes.  A row's sum (in ring_block.hip's order) would be a launch between the steps: the epilogue leaves the sums of
//     four neurons, at the next step each workgroup adds up and announces a row or two, and behind the products takes the
//     announced sums of all of its rows.  Nobody waits for one: what is not there yet is added up once more.  us per step with
//     a launch for operand and sums before each step -> here: N = 2048, 16 channels, B = 256: 57.9 -> 55.8; B = 1: 34.1 -> 29.7;
//     2 channels, B = 1: 11.4 -> 7.5; N = 2047, B = 16: 14.6 -> 8.9; N = 1500, 6 channels, B = 64: 15.0 -> 12.1.
//   * Around the products everything that waits for memory or LDS waits once, not once per row: the gates are loaded together, the
//     list of driven channels comes from sixteen channels at a time, a row tile's sum goes from wave to wave behind the tile
//     before it (and stays in registers where a workgroup has one column tile), the previous state is on its way meanwhile, the
//     announced row sums are asked for together.  At N = 2048, 16 channels, B = 256 these were 57 of the 130 thousand cycles of
//     a step, the products 72 (now some 30 and 60; the weights alone take 22 us to read, 6.6 TB/s).  us per step, T = 20 with
//     the packing launch: N = 2048, 16 channels, B = 256 66.2 -> 52.6, B = 1 35.2 -> 33.2; 12 channels, B = 1024 144 -> 111;
//     2 channels, B = 1024 48.8 -> 42.0; N = 1100, 16 channels, B = 1024 133 -> 94; N = 700, 6 channels, B = 1024 36.7 -> 28.7;
//     N = 1500, 6 channels, B = 64 14.4 -> 12.8.
// us per step, ring_block.hip / ring_bign.hip -> here, T = 20 with the packing launch:
//   N = 2048, 16 channels: B = 1: 120 -> 35   B = 256: 102 -> 63   B = 1024: 286 -> 181
//   N = 2048,  2 channels: B = 16: 31 -> 9    B = 256:  35 -> 19   B = 1024:  73 -> 44
//   N = 1100,  2 channels: B = 16: 22 -> 8.5  B = 200:  29 -> 17   N = 1500, 6 channels, B = 64: 49 -> 13
// Products, gates and activation are the arithmetic of ring_block.hip in the same order (a product's contraction is
// never split), so the two families agree bit for bit: tests/test_gpu_panel.py.
#include "ring_step_common.hpp"

namespace {

typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int PANEL_NV = 5;        // virtual columns per wave
constexpr int PANEL_S = 4;         // K chunks per LDS stage; weights are fetched two stages ahead

// What a pass over the contraction works on.  (All of it the same in every lane.)
struct PanelPass {
  __amdgpu_buffer_rsrc_t x, w;        // operand fragments, packed weights
  unsigned wat[PANEL_NV];             // byte offset of the wave's virtual columns, chunk 0
  int mat[PANEL_NV], col[PANEL_NV];   // their matrix and column tile
  const float* gl;       // gates [1 + k][16 R + 4], those of matrix 0 all J1
  int KCH, C, nv, wv;
};

// The previous state of the outputs a thread will form (four neurons of a row each): on its way while the products are summed,
// then in LDS (where the operand was), in the thread's own places.
template <int R>
struct PanelPrev {
  const float* prev;     // null: not behind this pass
  int N, B, C, first_row, first_col, tid;
};

// A fragment per lane from a scalar byte offset.  (Buffer loads: every address but the lane's own 16 bytes is scalar, which
// leaves the registers to the fragments in flight.)
__device__ __forceinline__ bf16x8 panel_load(__amdgpu_buffer_rsrc_t r, unsigned at, int lane) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (int)at, 0));
}

// The products X_i @ W_v of a wave's NV virtual columns with all row tiles, then gates and the sum over the matrices in
// their order into sums [C][R][64]: a row tile goes from wave to wave, the next one a barrier behind it.  (All of a wave's tiles
// before the next wave's took 28 of 136 thousand cycles at N = 2048, 16 channels, B = 256.)
template <int R, int NV>
__device__ __forceinline__ void panel_pass(const PanelPass& p, const unsigned (&xrow)[R], bf16x8* xs, f32x4* sums, int lane, const PanelPrev<R>& was) {
  const int KCH = p.KCH, nst = KCH / PANEL_S, wv = p.wv;
  auto stage = [&](int buf, int i, int d) { return xs + ((buf * R + i) * PANEL_S + d) * 64 + lane; };
  f32x4 acc[NV][R];
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < R; ++i) {
      acc[v][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[v][i]));                 // products live in the accumulation-register half
    }
  bf16x8 x0[R], xr[R], wf[2 * PANEL_S][NV], xa[2][R];
  // wave d carries chunk d of every row tile of a stage into LDS.  (The second stage's loads go out before the weights',
  // as in the loop: its wait at the top of the loop then leaves the weights in flight on both ways in.)
#pragma unroll
  for (int i = 0; i < R; ++i) x0[i] = panel_load(p.x, xrow[i] + wv * 1024, lane);
#pragma unroll
  for (int i = 0; i < R; ++i) xr[i] = panel_load(p.x, xrow[i] + (PANEL_S + wv) * 1024, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < 2 * PANEL_S; ++d)
#pragma unroll
    for (int v = 0; v < NV; ++v) wf[d][v] = panel_load(p.w, p.wat[v] + d * 1024, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    *stage(0, i, wv) = x0[i];
    asm volatile("" : "+v"(xr[i]));      // (used here, or the compiler moves the loads behind the weights')
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < R; ++i) xa[0][i] = *stage(0, i, 0);
#pragma unroll 1
  for (int s0 = 0; s0 < nst; s0 += 2)                     // (the number of stages is a multiple of four)
#pragma unroll
    for (int cur = 0; cur < 2; ++cur) {
      const int s = s0 + cur, nxt = cur ^ 1;
      const int sx = s + 2 < nst ? s + 2 : nst - 1;       // past the end: a re-read, unused
      // Memory and LDS instructions go out a few at a time behind the matrix instructions of a column: a burst of them, in all four
      // waves at once, keeps the one wave of a SIMD from issuing anything else (of 33 us of products at N = 2048, 16 channels,
      // B = 256 the matrix instructions alone take 20, the LDS reads 5 more, the loads 7).  us a call, T = 20, in bursts and so:
      // N = 2048, 16 channels, B = 256 913 -> 883, two of them driven 528 -> 497; T = 40: N = 1100, 8 channels, B = 600 1430 -> 1373,
      // N = 1500, 2 channels, B = 1000 1293 -> 1250.  One or two row tiles have too few instructions to hide behind (N = 2048, two of
      // 16 driven, B = 16, T = 40 408 -> 415): their loads go out together.
      constexpr bool SPREAD = R >= 4;
      auto next_x = [&](int i) {                          // (the barrier of the stage before: nobody reads that buffer any more)
        *stage(nxt, i, wv) = xr[i];
        xr[i] = panel_load(p.x, xrow[i] + (PANEL_S * sx + wv) * 1024, lane);
      };
      if constexpr (!SPREAD) {
#pragma unroll
        for (int i = 0; i < R; ++i) *stage(nxt, i, wv) = xr[i];
#pragma unroll
        for (int i = 0; i < R; ++i) xr[i] = panel_load(p.x, xrow[i] + (PANEL_S * sx + wv) * 1024, lane);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int d = 0; d < PANEL_S; ++d) {
        if (d + 1 == PANEL_S) lds_barrier();              // the next stage is in LDS; all reads of this one have landed
        auto next_xa = [&](int i) { xa[(d + 1) & 1][i] = d + 1 < PANEL_S ? *stage(cur, i, d + 1) : *stage(nxt, i, 0); };
        if constexpr (!SPREAD) {
#pragma unroll
          for (int i = 0; i < R; ++i) next_xa(i);
        }
        __builtin_amdgcn_sched_barrier(0);
        bf16x8(&w)[NV] = wf[PANEL_S * cur + d];
        // (past the end: re-reads, unused.  With eight row tiles not all of one chunk, whose lines would be waited for one after the
        // other: as a share of the time in bursts N = 1024, 16 channels, B = 256, T = 40 1.00 so, 0.97 with the last stage's chunks,
        // N = 1500, two of 16 driven, B = 130 0.95 and 0.935; with four the other way round: N = 2000, 12 channels, B = 60 1.00 and 1.01)
        const int kp = R == 8 ? PANEL_S * sx + d : PANEL_S * (s + 2) + d < KCH ? PANEL_S * (s + 2) + d : KCH - 1;
        auto next_w = [&](int v) { w[v] = panel_load(p.w, p.wat[v] + kp * 1024, lane); };
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          if constexpr (SPREAD) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = v * R / NV; i < (v + 1) * R / NV; ++i) next_xa(i);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int i = 0; i < R; ++i) acc[v][i] = mfma16(xa[d & 1][i], w[v], acc[v][i]);
          if constexpr (SPREAD) {
            __builtin_amdgcn_sched_barrier(0);
            next_w(v);
            if (d < 2) {
              const int at = d * NV + v;
#pragma unroll
              for (int i = at * R / (2 * NV); i < (at + 1) * R / (2 * NV); ++i) next_x(i);
            }
          }
        }
        if constexpr (!SPREAD) {
#pragma unroll
          for (int v = 0; v < NV; ++v) next_w(v);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  f32x4 prev[R];                         // (R C / 4 of them are used)
  if (was.prev) {
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int idx = was.tid + 256 * n, row = idx / (4 * was.C), j4 = 4 * (idx % (4 * was.C));
      if (idx < R * 16 * 4 * was.C) prev[n] = load4_masked(was.prev, was.N, was.B, was.first_row + row, was.first_col + j4);
    }
  }
#pragma unroll 1
  for (int r = 0; r < wv; ++r) lds_barrier();
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (p.nv > 0) {
      f32x4 g[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) g[v] = *reinterpret_cast<const f32x4*>(p.gl + p.mat[v] * (16 * R + 4) + 16 * i + 4 * (lane >> 4));
      f32x4* dst = sums + (p.col[0] * R + i) * 64 + lane;
      f32x4 s = *dst;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if (v > 0 && p.C > 1) {                           // (with one column tile the sum stays in registers)
          *dst = s;
          dst = sums + (p.col[v] * R + i) * 64 + lane;
          s = *dst;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = fmaf(g[v][e], acc[v][i][e], s[e]);
      }
      *dst = s;
    }
    lds_barrier();
  }
#pragma unroll 1
  for (int r = wv; r < 3; ++r) lds_barrier();
  if (was.prev) {
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int idx = was.tid + 256 * n;
      if (idx < R * 16 * 4 * was.C) reinterpret_cast<f32x4*>(xs)[idx] = prev[n];
    }
  }
}

// The sum of a row of a [B][N] state from its fours [N / 4], by 16 lanes: ring_block.hip's order, and ring_panel_operand_kernel's.
template <int EACH>                                       // loads in flight
struct PanelRowSum {
  float v[EACH];
  __device__ __forceinline__ void load(const float* fours, int N, int at) {       // (past the end: a re-read, not summed)
    const int last = (N - 1) >> 2;
#pragma unroll
    for (int i = 0; i < EACH; ++i) v[i] = fours[at + 16 * i < last ? at + 16 * i : last];
  }
  __device__ __forceinline__ void add(float& s, int N, int at) const {
    const int last = (N - 1) >> 2;
#pragma unroll
    for (int i = 0; i < EACH; ++i) s += at + 16 * i <= last ? v[i] : 0.f;
  }
};
__device__ __forceinline__ float panel_row_sum(const float* fours, int N, int sub) {
  float s = 0.f;
  for (int at = sub; 4 * at < N; at += 16 * 16) {
    PanelRowSum<16> some;
    some.load(fours, N, at);
    some.add(s, N, at);
  }
  return row16_sum_dpp(s);
}

// What travels between the steps, two of each but the row sums (three: the step before the last one's is emptied).  Only the
// first operand and row sums where they come from a launch of their own.
struct PanelState {
  bf16x8* x[2];         // operand fragments [batch tile][K chunk][lane]
  float* fours[2];      // [row][NPAD / 4]
  float* rs[3];         // [row]; PANEL_EMPTY: not announced yet
};
constexpr unsigned PANEL_EMPTY = 0xFFFFFFFFu;

// Four neurons of a row as bf16, at their place in the operand fragments.
__device__ __forceinline__ void panel_put(bf16x8* x, int KCH, int b, int j, const f32x4& v) {
  char* base = reinterpret_cast<char*>(x + (size_t)(b >> 4) * KCH * 64);
  const bf16x4 pk = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
  *reinterpret_cast<bf16x4*>(base + (size_t)((j >> 5) * 64 + ((j >> 3) & 3) * 16 + (b & 15)) * 16 + (j & 7) * 2) = pk;
}

}  // namespace

// Operand fragments [batch tile][K chunk][lane][8] and fp32 row sums of the initial state's rows; four rows per wave.  The
// sums run in the order of stage_rows (ring_step_common.hpp).  (Both fragment buffers, if there are two: the steps write no
// padding.)
__global__ __launch_bounds__(64) void ring_panel_operand_kernel(const float* __restrict__ prev, PanelState ps, int N, int B, int NPAD) {
  const int lane = threadIdx.x, row = 4 * (blockIdx.x & 3) + (lane >> 4), sub = lane & 15, bt = blockIdx.x >> 2;
  const int b = 16 * bt + row;
  float sum = 0.f;
  auto put = [&](int j, f32x4 v) {
    sum += (v[0] + v[1]) + (v[2] + v[3]);
    panel_put(ps.x[0], NPAD >> 5, b, j, v);
    if (ps.x[1]) panel_put(ps.x[1], NPAD >> 5, b, j, v);
  };
  // Sixteen loads in flight: one at a time this launch is all latency, 12.7 against 5 us.  Addresses are clamped into the
  // row; where N is no multiple of four, values that reach past its end are read as the row's last four and moved into
  // place (N = 2047, B = 16, 2 channels: 25 -> 17 us per step).  (NPAD is a multiple of 512; what lies past it is skipped.)
  const float* src = prev + (size_t)(b < B ? b : B - 1) * N;
  if ((N & 3) == 0) {
    for (int j0 = 4 * sub; j0 < NPAD; j0 += 16 * 64) {
      f32x4 v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = *reinterpret_cast<const f32x4*>(src + (j0 + 64 * i < N ? j0 + 64 * i : 0));
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = j0 + 64 * i;
        if (j < NPAD) put(j, b < B && j < N ? v[i] : f32x4{0.f, 0.f, 0.f, 0.f});
      }
    }
  } else {
    for (int j0 = 4 * sub; j0 < NPAD; j0 += 16 * 64) {
      f32x4 v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = j0 + 64 * i;
        v[i] = *reinterpret_cast<const f32x4_u*>(src + (j + 4 <= N ? j : N - 4));
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = j0 + 64 * i, sh = j + 4 <= N ? 0 : j + 4 - N;
        f32x4 r = v[i];
        if (sh & 2) { r[0] = r[2]; r[1] = r[3]; }
        if (sh & 1) { r[0] = r[1]; r[1] = r[2]; r[2] = r[3]; }
#pragma unroll
        for (int x = 0; x < 4; ++x) r[x] = b < B && j + x < N ? r[x] : 0.f;
        if (j < NPAD) put(j, r);
      }
    }
  }
  sum = row16_sum_dpp(sum);
  if (sub == 0) {
    ps.rs[0][b] = sum;
    if (ps.rs[1]) ps.rs[1][b] = __builtin_bit_cast(float, PANEL_EMPTY);
  }
}

// One step for R row tiles x C column tiles (16 consecutive neurons each).  Wpack: order 3 of ring_pack_weights_kernel.
// CARRY: with the next step's operand and the sums of its fours.
template <int ACT, int R, bool CARRY>
__global__ __launch_bounds__(256) void ring_panel_fwd_kernel(RingFwdArgs p, PanelState state, int NC, int C, int t, int xcd_map) {
  extern __shared__ __attribute__((aligned(16))) char panel_lds[];
  __shared__ int list[BN_GATE_KMAX + 1];
  __shared__ float row_sums[16 * R];
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int N = p.N, B = p.B, T = p.T, k = p.k, KCH = 2 * NC;
  bf16x8* const xs = reinterpret_cast<bf16x8*>(panel_lds);                                  // [2][R][PANEL_S][64]
  f32x4* const sums = reinterpret_cast<f32x4*>(xs + (size_t)2 * R * PANEL_S * 64);          // [C][R][64]
  float* const gl = reinterpret_cast<float*>(sums + (size_t)C * R * 64);                    // [1 + k][16 R + 4]
  constexpr int GS = 16 * R + 4;
  int rg, cb;
  step_block_coords(xcd_map, rg, cb);
  const int bt0 = rg * R;
  const bf16x8* const xfrag = state.x[CARRY ? t & 1 : 0];
  // this workgroup's share of the row sums (there are at least as many column blocks as row tiles: a row per 16 lanes at
  // most), announced to the others of its rows
  const int sum_row = cb + (int)gridDim.y * (tid >> 4), sum_b = 16 * bt0 + sum_row;
  const bool sums_row = CARRY && sum_row < 16 * R && sum_b < B;
  // (the widest panels, whose steps are long, have its loads in flight over the gates' at the price of a longer program:
  // N = 2048, 16 channels, B = 256: 57.7 -> 56.2 us per step, but 2 channels, B = 1: 7.6 -> 8.4)
  constexpr bool EARLY = R == 8;
  const float* const own_fours = CARRY ? state.fours[t & 1] + (size_t)sum_b * (16 * NC) : nullptr;
  float own_sum = 0.f;
  PanelRowSum<EARLY ? 32 : 1> own;                          // (N <= 2048)
  if (sums_row && t > 0) {
    if constexpr (EARLY) own.load(own_fours, N, tid & 15);
    else own_sum = panel_row_sum(own_fours, N, tid & 15);
  }

  // (R loads on their way at a time: memory is busy with other workgroups' weights, and a load takes long)
  for (int idx0 = tid; idx0 < R * 16 * k; idx0 += 256 * R) {
    float g[R];
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int idx = idx0 + 256 * n, row = idx / k, c = idx - row * k, b = 16 * bt0 + row;
      g[n] = p.A[((size_t)(idx < R * 16 * k && b < B ? b : 0) * T + t) * k + c];
    }
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int idx = idx0 + 256 * n, row = idx / k, c = idx - row * k;
      if (idx < R * 16 * k) gl[(1 + c) * GS + row] = 16 * bt0 + row < B ? g[n] : 0.f;
    }
  }
  for (int i = tid; i < 16 * R; i += 256) gl[i] = p.J1;
  for (int i = tid; i < C * R * 64; i += 256) sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (sums_row) {
    if constexpr (EARLY) {
      own.add(own_sum, N, tid & 15);
      own_sum = row16_sum_dpp(own_sum);
    }
    if ((tid & 15) == 0) {
      if (t > 0) __hip_atomic_store(state.rs[t % 3] + sum_b, own_sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      state.rs[(t + 1) % 3][sum_b] = __builtin_bit_cast(float, PANEL_EMPTY);
    }
  }
  lds_barrier();
  // matrices worth multiplying: Wo, and the channels that are not zero in all of the workgroup's rows
  // (four lanes a channel, sixteen channels at once)
  int nact = 1;
  if (tid == 0) list[0] = 0;
  for (int c0 = 0; c0 < k; c0 += 16) {
    const int c = c0 + (lane >> 2);
    bool nz = false;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(gl + (1 + (c < k ? c : 0)) * GS + 16 * i + 4 * (lane & 3));
      nz |= v[0] != 0.f || v[1] != 0.f || v[2] != 0.f || v[3] != 0.f;
    }
    unsigned long long any = __ballot(nz && c < k);
    any |= any >> 1;
    any = (any | any >> 2) & 0x1111111111111111ull;        // a bit per channel, that of its first lane
    if (wv == 0 && (any >> lane) & 1) list[nact + __popcll(any & ((1ull << lane) - 1))] = c + 1;
    nact += __popcll(any);
  }
  nact = __builtin_amdgcn_readfirstlane(nact);
  lds_barrier();

  unsigned xrow[R];
#pragma unroll
  for (int i = 0; i < R; ++i) xrow[i] = (unsigned)(bt0 + i < p.nbt ? bt0 + i : p.nbt - 1) * (unsigned)KCH * 1024u;   // (past the end: a re-read)
  PanelPass ps;
  ps.x = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16x8*>(xfrag), 0, (int)((unsigned)p.nbt * (unsigned)KCH * 1024u), 0x00020000);
  ps.w = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Wpack), 0, (int)((unsigned)(k + 1) * 4u * NC * KCH * 1024u), 0x00020000);
  ps.gl = gl;
  ps.C = C;
  ps.KCH = KCH;
  ps.wv = wv;
  const int cs = C == 4 ? 2 : C - 1;                      // C is 1, 2 or 4
  const int per_pass = (4 * PANEL_NV) >> cs;              // matrices per pass over the contraction
  const float* const prev = t == 0 ? p.r_init : p.hist + (size_t)(t - 1) * B * N;
  PanelPrev<R> was{nullptr, N, B, C, 16 * bt0, 16 * C * cb, tid};
  for (int m0 = 0; m0 < nact; m0 += per_pass) {
    const int nm = nact - m0 < per_pass ? nact - m0 : per_pass, V = nm << cs;
    const int v0 = wv * V / 4;
    ps.nv = (wv + 1) * V / 4 - v0;                        // this wave's run; matrices ascending
    int mats[PANEL_NV];
#pragma unroll
    for (int v = 0; v < PANEL_NV; ++v) mats[v] = list[m0 + ((v < ps.nv ? v0 + v : (ps.nv > 0 ? v0 : 0)) >> cs)];
#pragma unroll
    for (int v = 0; v < PANEL_NV; ++v) {
      const int u = v < ps.nv ? v0 + v : (ps.nv > 0 ? v0 : 0);
      ps.mat[v] = __builtin_amdgcn_readfirstlane(mats[v]);
      ps.col[v] = u & (C - 1);
      ps.wat[v] = ((unsigned)ps.mat[v] * 4u * NC + (unsigned)(cb * C + ps.col[v])) * (unsigned)KCH * 1024u;
    }
    was.prev = m0 + per_pass >= nact ? prev : nullptr;
    // (every variant passes the same number of barriers; a wave without a column of its own helps with the staging)
    switch (ps.nv) {
      case 5: panel_pass<R, 5>(ps, xrow, xs, sums, lane, was); break;
      case 4: panel_pass<R, 4>(ps, xrow, xs, sums, lane, was); break;
      case 3: panel_pass<R, 3>(ps, xrow, xs, sums, lane, was); break;
      case 2: panel_pass<R, 2>(ps, xrow, xs, sums, lane, was); break;
      default: panel_pass<R, 1>(ps, xrow, xs, sums, lane, was); break;
    }
  }

  // (step and thread as the compiler does not know them from above: what follows from them is not kept over the products)
  int now = t, me = tid;
  if constexpr (CARRY) {
    asm volatile("" : "+s"(now), "+v"(me));
    float rs[R];
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int b = 16 * bt0 + (me >> 4) + 16 * n;
      rs[n] = __hip_atomic_load(state.rs[now % 3] + (b < B ? b : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int row = (me >> 4) + 16 * n, b = 16 * bt0 + row, sub = me & 15;
      if (b >= B) break;
      float s = rs[n];
      if (__builtin_bit_cast(unsigned, s) == PANEL_EMPTY)                      // (the same in the row's 16 lanes)
        s = panel_row_sum(state.fours[now & 1] + (size_t)b * (16 * NC), N, sub);
      if (sub == 0) row_sums[row] = s;
    }
    lds_barrier();
  }

  // activation and leak; a thread takes four consecutive neurons of a row
  float* out = p.hist + (size_t)now * B * N;
  const float oma = 1.f - p.alpha;
  const float* sf = reinterpret_cast<const float*>(sums);
#pragma unroll
  for (int n = 0; n < R; ++n) {
    const int idx = me + 256 * n;
    if (idx >= R * 16 * 4 * C) break;
    const int row = idx / (4 * C), j4 = 4 * (idx % (4 * C)), cc = j4 >> 4, nn = j4 & 15;
    const int b = 16 * bt0 + row, j = 16 * C * cb + j4, i = row >> 4;
    if (b >= B || j >= N) continue;
    const f32x4 rp = reinterpret_cast<const f32x4*>(xs)[idx];
    const float js = p.J0 * (CARRY ? row_sums[row] : state.rs[0][b]);
    f32x4 rn;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float s = sf[((size_t)(cc * R + i) * 64 + ((row & 15) >> 2) * 16 + nn + x) * 4 + (row & 3)];
      float F, D;
      act_fast<ACT>(s + js, F, D);
      rn[x] = fmaf(p.alpha, F, oma * rp[x]);
    }
    store4_masked(out, N, B, b, j, rn);
    if (CARRY && now + 1 < T) {
#pragma unroll
      for (int x = 1; x < 4; ++x) rn[x] = j + x < N ? rn[x] : 0.f;
      panel_put(state.x[(now + 1) & 1], KCH, b, j, rn);
      state.fours[(now + 1) & 1][(size_t)b * (16 * NC) + (j >> 2)] = (rn[0] + rn[1]) + (rn[2] + rn[3]);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Launchers
// ------------------------------------------------------------------------------------------------
static size_t panel_lds_bytes(int R, int C, int k) {
  return (size_t)2 * R * PANEL_S * 1024 + (size_t)C * R * 1024 + (size_t)(R * 16 + 4) * (k + 1) * sizeof(float);
}

// Row tiles and column tiles of a workgroup.  Per K chunk a workgroup needs the longer of its matrix-pipe time
// (16 cycles an MFMA, the fullest wave's share) and its loads: a compute unit takes in some 16 bytes per cycle from the
// memory side of its L2, whatever is in flight (measured: 18 KiB a chunk on 128 compute units and 25 KiB on 256 both run
// at 15 to 17).  Workgroups beyond one per compute unit queue.  us per step, N = 2048, by (row tiles, column tiles), with
// a launch for the operand of 5 us in each:
//   16 channels, B = 256:  (8,1) 64  (4,1) 71  (4,2) 66  (8,2) 98      B = 1:  (1,1) 39  (4,1) 45  (8,1) 57
//   16 channels, B = 1024: (8,1) 208 (8,2) 195 (8,4) 189               2 channels, B = 256:  (4,2) 22  (8,1) 27  (8,4) 43
static float panel_shape(int NC, int nbt, int k, int* R_out, int* C_out) {
  float best = 0.f, step = 0.f;
  for (int R = 1; R <= 8; R *= 2)
    for (int C = 1; C <= 4; C *= 2) {
      const int V = (k + 1) * C;
      if (R > 1 && R / 2 >= nbt) continue;
      if (panel_lds_bytes(R, C, k) > 150 * 1024) continue;
      const int passes = (V + 4 * PANEL_NV - 1) / (4 * PANEL_NV), Vp = (V + passes - 1) / passes;
      const long wgs = (long)((nbt + R - 1) / R) * (4 * NC / C), rounds = (wgs + 255) / 256;
      const float mfma = 16.f * (float)(((Vp + 3) / 4) * R), load = 1024.f * (float)(R + Vp) / 16.f;
      const float cost = (float)(rounds * passes) * (mfma > load ? mfma : load);
      if (best == 0.f || cost <= best) {      // (a tie goes to the wider panel: fewer workgroups fetch the same rows)
        best = cost;
        *R_out = R;
        *C_out = C;
        step = 0.72f * 2.f * NC * cost + (float)(rounds * passes * (R - 4)) * 2500.f + 14300.f;
      }
    }
  return step;
}

// Cycles of a step at 2.4 GHz, launch included, as fitted to 165 measured shapes (N = 640 to 2048, 2 to 16 channels, B = 4 to 1024:
// mean deviation 8 %, largest 27 %).
float ring_panel_step_cycles(int NC, int nbt, int k) {
  int R, C;
  return panel_shape(NC, nbt, k, &R, &C);
}

bool ring_panel_applicable(int NC, int k) { return NC >= 16 && NC % 8 == 0 && k <= BN_GATE_KMAX; }

static size_t panel_operand_bytes(int NC, int nbt) { return (size_t)nbt * 2 * NC * 1024; }
size_t ring_panel_workspace_bytes(int NC, int nbt) {
  return 2 * panel_operand_bytes(NC, nbt) + 2 * (size_t)nbt * 16 * 16 * NC * sizeof(float) + 3 * (size_t)nbt * 16 * sizeof(float);
}

// RINGATTR_PANEL=0: never; a switch that asks for one of the other step-per-launch families is obeyed.
bool ring_uses_panel(int k, int NC, int nbt) {
  if (!ring_panel_applicable(NC, k)) return false;
  const char* v = getenv("RINGATTR_PANEL");
  if (v && v[0] == '0') return false;
  for (const char* name : {"RINGATTR_WIDE", "RINGATTR_BLOCK", "RINGATTR_BLOCK_SHAPE"})
    if (getenv(name)) return false;
  return panel_operand_bytes(NC, nbt) < ((size_t)1 << 30);   // (32-bit offsets; the weights are 0.6 GB at most)
}

template <int ACT, int R, bool CARRY>
static hipError_t panel_steps(const RingFwdArgs& a, int NC, int C, hipStream_t st) {
  const size_t dyn = panel_lds_bytes(R, C, a.k);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ring_panel_fwd_kernel<ACT, R, CARRY>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
  if (e != hipSuccess) return e;
  PanelState ps = {};
  char* ws = reinterpret_cast<char*>(a.panel_ws);
  for (int i = 0; i < 2; ++i, ws += panel_operand_bytes(NC, a.nbt)) ps.x[i] = reinterpret_cast<bf16x8*>(ws);
  for (int i = 0; i < 2; ++i, ws += (size_t)a.nbt * 16 * 16 * NC * sizeof(float)) ps.fours[i] = reinterpret_cast<float*>(ws);
  for (int i = 0; i < 3; ++i, ws += (size_t)a.nbt * 16 * sizeof(float)) ps.rs[i] = reinterpret_cast<float*>(ws);
  if (!CARRY) ps.x[1] = nullptr, ps.rs[1] = nullptr;
  const dim3 grid((a.nbt + R - 1) / R, 4 * NC / C);
  const int xm = step_xcd_map();
  for (int t = 0; t < a.T; ++t) {
    if (t == 0 || !CARRY)
      RING_LAUNCH(ring_panel_operand_kernel, dim3(4 * a.nbt), dim3(64), 0, st, t == 0 ? a.r_init : a.hist + (size_t)(t - 1) * a.B * a.N, ps,
                  a.N, a.B, 64 * NC);
    RING_LAUNCH((ring_panel_fwd_kernel<ACT, R, CARRY>), grid, dim3(256), dyn, st, a, ps, NC, C, t, xm);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Where workgroups queue, a step's first ones find no announced sums (who would announce them has not begun) and add up all of
// their rows: with more than one a compute unit, operand and sums are a launch's.  us per step, carried and with the launch,
// N = 1100, 16 channels: B = 1000 146 and 133, B = 3000 444 and 385; N = 2048, one channel, B = 3000 126 and 110; with one a
// compute unit, N = 2048, B = 1000: one channel 39 and 41, 16 channels 191 and 193.  A single step has nothing to carry either
// (us a call: N = 1024, 5 channels, B = 512 36.2 and 33.2).
template <int ACT, int R>
static hipError_t panel_run(const RingFwdArgs& a, int NC, int C, hipStream_t st) {
  const bool queue = (long)((a.nbt + R - 1) / R) * (4 * NC / C) > 256;
  return queue || a.T == 1 ? panel_steps<ACT, R, false>(a, NC, C, st) : panel_steps<ACT, R, true>(a, NC, C, st);
}

template <int ACT>
static hipError_t panel_act(const RingFwdArgs& a, int NC, hipStream_t st) {
  int R = 1, C = 1;
  panel_shape(NC, a.nbt, a.k, &R, &C);
  if (const char* v = getenv("RINGATTR_PANEL_SHAPE")) {   // <R><C>, e.g. 81 (cross-checks)
    const int r = v[0] - '0', c = v[0] ? v[1] - '0' : 0;
    if ((r == 1 || r == 2 || r == 4 || r == 8) && (c == 1 || c == 2 || c == 4) && panel_lds_bytes(r, c, a.k) <= 150 * 1024) {
      R = r;
      C = c;
    }
  }
  switch (R) {
    case 8: return panel_run<ACT, 8>(a, NC, C, st);
    case 4: return panel_run<ACT, 4>(a, NC, C, st);
    case 2: return panel_run<ACT, 2>(a, NC, C, st);
    default: return panel_run<ACT, 1>(a, NC, C, st);
  }
}

// a.panel_ws: ring_panel_workspace_bytes; a.Wpack in order 3 of ring_pack_weights_kernel
hipError_t ring_launch_panel_fwd(const RingFwdArgs& a, int NC, hipStream_t st) {
  if (!ring_panel_applicable(NC, a.k) || !a.panel_ws || !a.hist || a.dfrag || a.rfrag) return hipErrorInvalidValue;
  switch (a.act) {
    case ACT_RELU: return panel_act<ACT_RELU>(a, NC, st);
    case ACT_GELU: return panel_act<ACT_GELU>(a, NC, st);
    case ACT_TANH: return panel_act<ACT_TANH>(a, NC, st);
    case ACT_SILU: return panel_act<ACT_SILU>(a, NC, st);
    default: return hipErrorInvalidValue;
  }
}
