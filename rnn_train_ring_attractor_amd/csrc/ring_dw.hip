// Weight-gradient contraction, register-tiled, for NPAD >= 128.
//
//   dW_mm[i][j] = sum over samples (b,t) of coef_mm(b,t) * g[t,b,i] * r_prev[t,b,j]
//
// A workgroup (4 waves, one per SIMD) owns a 128 (i) x 128 (j) block of up to three matrices over one
// K split; wave v owns rows 32v..32v+31 against all 128 columns: 2 x 8 MFMA tiles x 3 matrices = 48
// accumulators (192 accumulation VGPRs).  A K chunk is 16 batch rows x 2 time steps (32 samples, one
// MFMA K).  The paired tile-major operand buffers hold every tile of a chunk as 1 KiB of ready-made
// MFMA fragments, so nothing is ever transposed or repacked:
//   * the wave's own two g fragments load straight into registers;
//   * the action gates of a chunk (16 rows x 2 steps x up to 3 matrices) are fetched one value per
//     thread and handed round through a small LDS stage next to the r_prev one: per-lane gate loads
//     (eight scattered 4-byte loads per wave and chunk) cost more than the whole gating arithmetic;
//   * the eight r_prev fragments every wave needs are copied verbatim into an LDS stage of DW_LDS
//     buffers once per workgroup (8 KiB per chunk) and read back with conflict-free ds_read_b128, one
//     chunk ahead of the MFMAs that use them -- L2 -> CU traffic stays at 16 KiB per chunk and the LDS
//     pipe at 40 KiB, both under the MFMA time.
// DW_DEPTH chunks are in flight in registers; a trip of the main loop is one basic block containing
// loads only, so the compiler waits for exactly the oldest chunk (s_waitcnt vmcnt(n), n > 0).
// Partials are written once per wave; a fixed-order reduction follows.
#include "ring_common.hpp"
#include "ring_kernels.hpp"

#include <stdlib.h>

#include <utility>

namespace {

constexpr int DW_WI = 2;      // MFMA row tiles per wave (32 neurons of g)
constexpr int DW_WJ = 8;      // MFMA column tiles per wave (128 neurons of r_prev)
constexpr int DW_DEPTH = 4;   // K chunks in flight per wave
constexpr int DW_LDS = 4;     // LDS stage buffers (chunk c lives in buffer c % DW_LDS)

template <int NG>
struct DwStage {
  bf16x8 a[DW_WI];                    // g fragments of the wave's row tiles
  f32x4 bpart[2];                     // this thread's two fragments of the chunk's r_prev block (LDS stage)
  float gate;                         // one action gate of the chunk: matrix tid/32 % 4, row (tid/2) % 16, step tid % 2
};

// The order of a chunk's instructions around its N matrix instructions.  A SIMD has one wave here, and what that wave issues in a row
// (twelve LDS reads, the fifteen vector instructions of a gated fragment, five loads, the LDS stage) keeps its matrix pipe waiting: 1575
// cycles a chunk for 768 of products.  So a matrix instruction is followed by at most one of READS LDS reads, WRITES LDS writes, LOADS
// loads (behind the last uses of what they replace) and two vector instructions, which cost it nothing: 1345 cycles a chunk (N = 256,
// 15360 chunks; vector beside matrix instructions in 66.8 instead of 28.6 million of 189 million matrix cycles).  us of contraction, left to the
// compiler and so (same bits): N = 256, 15360 chunks 229 -> 194; N = 512, 12800 chunks 622 -> 517; N = 1024, 3840 chunks 690 -> 610.
// By vector instructions behind each: N = 512 three 560, two and three in turn 543 to 552, two 521 to 530, one 615.
template <int N, int READS, int WRITES, int LOADS, int I>
__device__ __forceinline__ void dw_spread_one() {
  constexpr int MFMA = 0x008, VALU = 0x002, VMEM_READ = 0x020, DS_READ = 0x100, DS_WRITE = 0x200, LATE = N - LOADS - 3;
  __builtin_amdgcn_sched_group_barrier(MFMA, 1, 0);
  if constexpr (I < READS) __builtin_amdgcn_sched_group_barrier(DS_READ, 1, 0);
  if constexpr (I >= READS + 2 && I < READS + 2 + WRITES) __builtin_amdgcn_sched_group_barrier(DS_WRITE, 1, 0);
  __builtin_amdgcn_sched_group_barrier(VALU, 2, 0);
  if constexpr (I >= LATE && I < LATE + LOADS) __builtin_amdgcn_sched_group_barrier(VMEM_READ, 1, 0);
}
template <int READS, int WRITES, int LOADS, int... I>
__device__ __forceinline__ void dw_spread(std::integer_sequence<int, I...>) {
  (dw_spread_one<(int)sizeof...(I), READS, WRITES, LOADS, I>(), ...);
}

// NMAT matrices in this launch's group, the first of them ungated (Wo) when FIRST.
// ga points at this lane's fragment of the wave's first row tile, rb at fragment `tid` of the block's
// eight column tiles (512 fragments, two per thread); chunks are laid out back to back (pair-major,
// batch tile fastest), 4*NC KiB apart.
template <int NC, int NMAT, bool FIRST>
__device__ __forceinline__ void dw_fetch(const RingDwArgs& p, const bf16x8* ga, const f32x4* rb, int bt, int t0, int mg,
                                         int tid, DwStage<NMAT - (FIRST ? 1 : 0)>& s) {
  const int T = p.T, k = p.k;
#pragma unroll
  for (int u = 0; u < DW_WI; ++u) s.a[u] = ga[u * 64];
  s.bpart[0] = rb[0];
  s.bpart[1] = rb[256];
  // gate of (gated matrix ga, sample row, step t0 + tt) for thread tid = 32*ga + 2*row + tt (mod 128).
  // The address is clamped into the tensor and the value used as loaded: rows past B and the missing
  // second step of an odd-length sequence meet zero g fragments.
  {
    const int gi = tid & 127, gm = gi >> 5, row = (gi >> 1) & 15, tt = gi & 1;
    constexpr int NG = NMAT - (FIRST ? 1 : 0);
    const int ch = 3 * mg + (gm < NG ? gm : 0) - (FIRST ? 0 : 1);   // matrix 3*mg + a gates with channel 3*mg + a - 1
    const int b = 16 * bt + row, bc = b < p.B ? b : p.B - 1;
    const int tg = t0 + tt < T ? t0 + tt : t0;
    s.gate = p.A[((size_t)bc * T + tg) * k + ch];
  }
}

// g8 = gates of rows 4q..4q+3 as (t0, t0+1) pairs: K slot e of the fragment is row e at t0, slot 4+e row e at t0+1
__device__ __forceinline__ bf16x8 gate_frag(bf16x8 x, const f32x4 (&g8)[2]) {
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[e] = (__bf16)((float)x[e] * g8[e >> 1][2 * (e & 1)]);
    o[4 + e] = (__bf16)((float)x[4 + e] * g8[e >> 1][2 * (e & 1) + 1]);
  }
  return o;
}

// ------------------------------------------------------------------------------------------------
// Short contractions: the four waves of a workgroup share out its K chunks instead of its rows.
// ------------------------------------------------------------------------------------------------
// What bounds a few hundred chunks is not the products: with a 128 x 128 block per workgroup the chip is only filled by many
// K splits, and a split's partial sums (64 KiB a matrix and block) are written and read once more.  Here a workgroup has a
// 32 x 128 block (a quarter of it), its wave w every fourth chunk from the w-th on, and the waves' sums are added in LDS: for
// the same number of workgroups a quarter of the splits and of the partial sums.  Blocks past the ring's own tiles are not
// there at all, and a launch takes up to four matrices (256 accumulation registers).  No barrier and no LDS stage: each wave
// loads its ten fragments of a chunk, DWS_DEPTH chunks ahead; the gates go from lane to lane through a wave's own LDS.
// us of contraction and reduction, with 128 x 128 blocks and here: N = 120, 2 channels, 240 chunks 20.2 -> 13.4; N = 256, 2 channels,
// 400 chunks 25.8 -> 16.4; N = 360, 3 channels, 266 chunks (two launches there) 48.9 -> 22.9.
constexpr int DWS_DEPTH = 3;

template <int NG>
struct DwChunk {
  bf16x8 a[DW_WI], b[DW_WJ];
  float gate[NG > 2 ? 2 : 1];           // (matrix, row, step) number lane (+ 64) of the chunk
};

// Tiles per side that hold neurons of the ring.
__host__ __device__ __forceinline__ int dw_tiles(const RingDwArgs& p, int NT) {
  const int group = p.linear_tiles ? 1 : NT / 4;          // (NT / 4 consecutive tiles share 4 NT neurons)
  return (p.N + 16 * group - 1) / (16 * group) * group;
}

template <int NMAT, bool FIRST>
__device__ __forceinline__ void dw_chunk_waves(const RingDwArgs& p, int m0, int NT) {
  constexpr int NG = NMAT - (FIRST ? 1 : 0), NLD = NG > 2 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4 sums[4][DW_WJ][64];
  __shared__ __attribute__((aligned(16))) float gates[4][DWS_DEPTH][4][16][2];     // [wave][stage][gated matrix][row][step]
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int tiles = dw_tiles(p, NT), ni = (tiles + DW_WI - 1) / DW_WI, nb = ni * ((tiles + DW_WJ - 1) / DW_WJ);
  // The workgroups of a K split read the same chunks: in the order in which the XCDs (dealt out round robin) hold consecutive
  // workgroups, so that a split is on as few as can be.
  const int at = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3), z = at / nb, block = at % nb;
  if (z >= p.nz) return;
  const int it0 = (block % ni) * DW_WI, jt0 = (block / ni) * DW_WJ;
  const int T = p.T, k = p.k, nbt = p.nbt;
  const int nchunk = nbt * ((T + 1) / 2);                 // (the host checked that it fits an int)
  const int ch0 = (int)((long)nchunk * z / p.nz) + wv, ch1 = (int)((long)nchunk * (z + 1) / p.nz);
  const int n = ch0 < ch1 ? (ch1 - ch0 + 3) / 4 : 0;

  f32x4 acc[NMAT][DW_WI][DW_WJ];
#pragma unroll
  for (int a = 0; a < NMAT; ++a)
#pragma unroll
    for (int ii = 0; ii < DW_WI; ++ii)
#pragma unroll
      for (int u = 0; u < DW_WJ; ++u) {
        acc[a][ii][u] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[a][ii][u]));
      }

  // the fetch cursor parks on the wave's last chunk, as above (a wave without any: on some chunk)
  const int first = ch0 < nchunk ? ch0 : nchunk - 1;
  const size_t step = (size_t)4 * NT * 64;
  const bf16x8* ga = reinterpret_cast<const bf16x8*>(p.gfrag) + ((size_t)first * NT + it0) * 64 + lane;
  const bf16x8* rb = reinterpret_cast<const bf16x8*>(p.rfrag) + ((size_t)first * NT + jt0) * 64 + lane;
  int left = n, fb = first % nbt, ft = first / nbt;
  const int db = 4 % nbt, dt = 4 / nbt;
  const int row = (lane >> 1) & 15, tt = lane & 1;
  auto fetch = [&](DwChunk<NG>& s) {
#pragma unroll
    for (int u = 0; u < DW_WI; ++u) s.a[u] = ga[u * 64];
#pragma unroll
    for (int u = 0; u < DW_WJ; ++u) s.b[u] = rb[u * 64];
    // rows past B and the missing second step of an odd-length sequence meet zero g fragments: any gate will do there
    const int b = 16 * fb + row, bc = b < p.B ? b : p.B - 1, tg = 2 * ft + tt < T ? 2 * ft + tt : 2 * ft;
#pragma unroll
    for (int v = 0; v < NLD; ++v) {
      const int gm = 2 * v + (lane >> 5), ch = m0 + (gm < NG ? gm : 0) - (FIRST ? 0 : 1);
      s.gate[v] = NG > 0 ? p.A[((size_t)bc * T + tg) * k + ch] : 0.f;
    }
    const int adv = left > 1 ? 1 : 0;
    left -= adv;
    ga += adv * step;                                    // (products: a select of all of these would become a branch)
    rb += adv * step;
    fb += adv * db;
    ft += adv * dt;
    const int wrap = fb >= nbt ? 1 : 0;
    fb -= wrap * nbt;
    ft += wrap;
  };
  auto publish = [&](const DwChunk<NG>& s, int buf) {
    if constexpr (NG > 0)
#pragma unroll
      for (int v = 0; v < NLD; ++v) (&gates[wv][buf][0][0][0])[64 * v + lane] = s.gate[v];
  };
  // What a wave's lanes put into its LDS, other lanes of it read behind this.  (No instruction: a wave's LDS accesses are carried out in
  // order; it is the compiler that must not move one past the other.)
  auto handed_over = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto compute = [&](const DwChunk<NG>& s, int buf) {
    f32x4 g8[NG > 0 ? NG : 1][2];
#pragma unroll
    for (int a = 0; a < NG; ++a) {
      const f32x4* gp = reinterpret_cast<const f32x4*>(&gates[wv][buf][a][4 * (lane >> 4)][0]);
      g8[a][0] = gp[0];
      g8[a][1] = gp[1];
    }
#pragma unroll
    for (int a = 0; a < NMAT; ++a)
#pragma unroll
      for (int ii = 0; ii < DW_WI; ++ii) {
        const bf16x8 gg = (FIRST && a == 0) ? s.a[ii] : gate_frag(s.a[ii], g8[a - (FIRST ? 1 : 0)]);
#pragma unroll
        for (int u = 0; u < DW_WJ; ++u) acc[a][ii][u] = mfma16(gg, s.b[u], acc[a][ii][u]);
      }
  };
  DwChunk<NG> st[DWS_DEPTH];
#pragma unroll
  for (int d = 0; d < DWS_DEPTH; ++d) {
    fetch(st[d]);
    __builtin_amdgcn_sched_barrier(0);
  }
  publish(st[0], 0);
  handed_over();
  int i = 0;
#pragma unroll 1
  for (; i + DWS_DEPTH <= n; i += DWS_DEPTH)
#pragma unroll
    for (int d = 0; d < DWS_DEPTH; ++d) {
      compute(st[d], d);
      fetch(st[d]);
      publish(st[(d + 1) % DWS_DEPTH], (d + 1) % DWS_DEPTH);
      dw_spread<2 * NG, (NG > 0 ? NLD : 0), DW_WI + DW_WJ + NLD>(std::make_integer_sequence<int, NMAT * DW_WI * DW_WJ>{});
      handed_over();
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int d = 0; d < DWS_DEPTH - 1; ++d) {              // what is left: in stages 0 ...
    if (i + d >= n) break;
    compute(st[d], d);
    publish(st[d + 1], d + 1);
    handed_over();
  }

  // the waves' sums, in wave order; wave w writes out columns 2w and 2w + 1
#pragma unroll
  for (int a = 0; a < NMAT; ++a)
#pragma unroll
    for (int ii = 0; ii < DW_WI; ++ii) {
      lds_barrier();
#pragma unroll
      for (int u = 0; u < DW_WJ; ++u) sums[wv][u][lane] = acc[a][ii][u];
      lds_barrier();
#pragma unroll
      for (int uu = 0; uu < 2; ++uu) {
        const int u = 2 * wv + uu;
        const f32x4 s = ((sums[0][u][lane] + sums[1][u][lane]) + sums[2][u][lane]) + sums[3][u][lane];
        p.partial[((((size_t)z * (k + 1) + m0 + a) * NT + it0 + ii) * NT + jt0 + u) * 64 + lane] = s;
      }
    }
}

}  // namespace

// seg_begin / seg_end: the launch covers K chunks [seg_begin, seg_end) of the sequence (chunk = time-step pair *
// batch tiles + batch tile, so a range of chunks is a range of time steps); add != 0: the wave adds its result
// to the partial sums an earlier launch left.  NC = 0: dw_chunk_waves, of matrices mg ... at NT = seg_begin tiles a side.
template <int NC, int NMAT, bool FIRST>
__global__ __launch_bounds__(256) void ring_dw_direct_kernel(RingDwArgs p, int mg, int seg_begin, int seg_end, int add) {
  if constexpr (NC == 0) {
    dw_chunk_waves<NMAT, FIRST>(p, mg, seg_begin);
    return;
  } else {
  constexpr int NT = 4 * NC;
  constexpr int NB = NT / 8;             // 128-neuron blocks per side
  constexpr int NG = NMAT - (FIRST ? 1 : 0);
  __shared__ __attribute__((aligned(16))) f32x4 lds_b[DW_LDS][DW_WJ * 64];
  __shared__ __attribute__((aligned(16))) float lds_g[DW_LDS][8][16][2];   // [buffer][gated matrix, twice][row][step]
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int tiles = NB * NB;
  // keep the workgroups that share a K split on one XCD (workgroup ids are dealt round-robin to
  // the 8 XCDs) so the operand bytes they all read come out of that XCD's L2
  int z, tile;
  {
    const int bid = blockIdx.x;
    if ((p.nz & 7) == 0) {
      const int xcd = bid & 7, slot = bid >> 3;
      z = xcd * (p.nz >> 3) + slot / tiles;
      tile = slot % tiles;
    } else {
      z = bid / tiles;
      tile = bid % tiles;
    }
  }
  const int it0 = (tile % NB) * 8 + wv * DW_WI;
  const int jt0 = (tile / NB) * 8;

  const int nchunk = seg_end - seg_begin;       // (the host checked that the sequence's chunk count fits an int)
  const int ch0 = seg_begin + (int)((long)nchunk * z / p.nz), ch1 = seg_begin + (int)((long)nchunk * (z + 1) / p.nz);

  f32x4 acc[NMAT][DW_WI][DW_WJ];
#pragma unroll
  for (int a = 0; a < NMAT; ++a)
#pragma unroll
    for (int ii = 0; ii < DW_WI; ++ii)
#pragma unroll
      for (int u = 0; u < DW_WJ; ++u) {
        acc[a][ii][u] = f32x4{0.f, 0.f, 0.f, 0.f};
        // accumulate in the accumulation-VGPR half of the register file; the architectural half
        // then holds nothing but the operand stages in flight
        asm volatile("" : "+a"(acc[a][ii][u]));
      }

  // Fetch cursor: chunk = (batch tile fb, time-step pair ft), batch tile fastest.  It advances with
  // scalar selects (no branch, no division) and parks on the last chunk of the split, so fetches
  // past the end re-read valid data that is never consumed.
  int fc = ch0, fb = ch0 % p.nbt, ft = ch0 / p.nbt;
  constexpr size_t CHUNK_FRAGS = (size_t)NT * 64;   // 16-byte fragments per chunk
  const bf16x8* ga = reinterpret_cast<const bf16x8*>(p.gfrag) + (size_t)ch0 * CHUNK_FRAGS + (size_t)it0 * 64 + lane;
  const f32x4* rb = reinterpret_cast<const f32x4*>(p.rfrag) + (size_t)ch0 * CHUNK_FRAGS + (size_t)jt0 * 64 + tid;
  auto fetch_next = [&](DwStage<NG>& s) {
    dw_fetch<NC, NMAT, FIRST>(p, ga, rb, fb, 2 * ft, mg, tid, s);
    const int adv = (fc + 1 < ch1) ? 1 : 0;
    ga += adv * CHUNK_FRAGS;
    rb += adv * CHUNK_FRAGS;
    fc += adv;
    fb += adv;
    const int wrap = (fb == p.nbt) ? 1 : 0;
    fb = wrap ? 0 : fb;
    ft += wrap;
  };
  // The LDS stage has DW_LDS buffers and is read one chunk ahead of the MFMAs that use it: the reads of
  // chunk i+1 are issued before the MFMAs of chunk i and land while those run.  A chunk is therefore
  // published two chunks before it is used, with a barrier between the publication and the read.
  struct DwOperands {
    bf16x8 b[DW_WJ];
    f32x4 g8[NG > 0 ? NG : 1][2];
  };
  auto lds_read = [&](DwOperands& o, int buf) {
#pragma unroll
    for (int u = 0; u < DW_WJ; ++u) o.b[u] = *reinterpret_cast<const bf16x8*>(&lds_b[buf][u * 64 + lane]);
#pragma unroll
    for (int a = 0; a < NG; ++a) {
      const f32x4* gp = reinterpret_cast<const f32x4*>(&lds_g[buf][a][4 * (lane >> 4)][0]);
      o.g8[a][0] = gp[0];
      o.g8[a][1] = gp[1];
    }
  };
  auto compute = [&](const DwStage<NG>& s, const DwOperands& o) {
#pragma unroll
    for (int a = 0; a < NMAT; ++a) {
#pragma unroll
      for (int ii = 0; ii < DW_WI; ++ii) {
        const bf16x8 gg = (FIRST && a == 0) ? s.a[ii] : gate_frag(s.a[ii], o.g8[a - (FIRST ? 1 : 0)]);
#pragma unroll
        for (int u = 0; u < DW_WJ; ++u) acc[a][ii][u] = mfma16(gg, o.b[u], acc[a][ii][u]);
      }
    }
  };
  auto publish = [&](const DwStage<NG>& s, int buf) {
    lds_b[buf][tid] = s.bpart[0];
    lds_b[buf][tid + 256] = s.bpart[1];
    (&lds_g[buf][0][0][0])[tid] = s.gate;               // (no branch: the loop is one block to schedule)
  };

  if (ch0 < ch1) {
    static_assert(DW_DEPTH == DW_LDS, "stage d of the register pipeline and LDS buffer d hold the same chunk");
    DwStage<NG> st[DW_DEPTH];
    DwOperands op[2];
#pragma unroll
    for (int d = 0; d < DW_DEPTH; ++d) fetch_next(st[d]);
    publish(st[0], 0);
    publish(st[1], 1);
    lds_barrier();
    lds_read(op[0], 0);
    // Invariant at the top of step d (chunk base + d): op[d & 1] holds (or is about to receive) that chunk's
    // operands, buffer d + 1 holds the next chunk behind a barrier, stage d + 2 is the next to publish.
    int base = ch0;
    for (; base + DW_DEPTH <= ch1; base += DW_DEPTH) {
#pragma unroll
      for (int d = 0; d < DW_DEPTH; ++d) {
        lds_read(op[(d + 1) & 1], (d + 1) % DW_LDS);
        compute(st[d], op[d & 1]);
        fetch_next(st[d]);                          // refill DW_DEPTH chunks ahead
        publish(st[(d + 2) % DW_DEPTH], (d + 2) % DW_LDS);
        dw_spread<DW_WJ + 2 * NG, 3, 5>(std::make_integer_sequence<int, NMAT * DW_WI * DW_WJ>{});
        lds_barrier();
        // keep the refill of stage d where it is: the scheduler would otherwise sink all refills of
        // a trip to its end and drain the whole queue once per trip
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // tail (< DW_DEPTH chunks): stage d holds chunk base + d (past the split's end: copies of its last chunk)
#pragma unroll
    for (int d = 0; d < DW_DEPTH - 1; ++d) {
      if (base + d >= ch1) break;
      lds_read(op[(d + 1) & 1], (d + 1) % DW_LDS);
      compute(st[d], op[d & 1]);
      publish(st[(d + 2) % DW_DEPTH], (d + 2) % DW_LDS);
      lds_barrier();
    }
  }

#pragma unroll
  for (int a = 0; a < NMAT; ++a) {
    const int mm = 3 * mg + a;
#pragma unroll
    for (int ii = 0; ii < DW_WI; ++ii)
#pragma unroll
      for (int u = 0; u < DW_WJ; ++u) {
        ring_f32x4* dst = p.partial + ((((size_t)z * (p.k + 1) + mm) * NT + it0 + ii) * NT + jt0 + u) * 64 + lane;
        *dst = add ? *dst + acc[a][ii][u] : acc[a][ii][u];
      }
  }
  }
}

// N <= 128: a launch per three matrices, of a few workgroups where there is little to contract, against one launch for all
// matrices of the kernel with a wave per 32 x 128 block.  A training pass on this kernel, as a share of its time on that one,
// N = 65 to 128, by launches and chunks of the contraction (16 rows x two steps):
//   two launches    10: 1.07-1.10   50: 1.03-1.07   64: 0.90-0.98   128: 0.84-0.95   440: 0.95-0.99
//   three           10: 1.14-1.18   50: 1.11-1.14   64: 1.02-1.09   88: 0.99-1.03   128: 0.94-0.98   440: 0.90-0.94
//   four            10: 1.19-1.20   64: 1.15-1.20   88: 1.04-1.08   128: 0.96-1.00   440: 0.96-0.98
//   five and six    10: 1.22-1.26   64: 1.18-1.31   128: 1.05-1.12   190: 1.05-1.08   440: 0.96-0.98
//   nine            480: 0.99   960: 1.00
// Up to two channels there is one launch here too.
bool ring_dw_tiled_applicable(int NC, int k, long nchunk) {
  const int launches = (k + 3) / 3;
  if (NC == 2) return launches == 1 || nchunk > (launches == 2 ? 56 : launches == 3 ? 96 : launches == 4 ? 112 : launches <= 6 ? 256 : 512);
  return NC == 4 || NC == 8 || NC == 16 || NC == 24 || NC == 32;
}

// K splits: one workgroup per CU, a multiple of 8 when possible (XCD grouping).  One launch per
// group of three matrices, so the grid of a launch does not depend on a_dim.
// N <= 128 (one block): a split's partial sums are 64 KiB a matrix, as much to write and to sum up as some four chunks take to
// contract, so none gets fewer, and with more than five channels there are at most 80 splits.  us of contraction and
// reduction against a wave per 32 x 128 block without an LDS stage: N = 120, a_dim 2, T = 240, B = 64 33 -> 25, B = 4096
// 932 -> 123.
int ring_dw_tiled_nz(int NC, int k, long nchunk) {
  const int NB = 4 * NC / 8;
  const long tiles = (long)NB * NB;
  long nz = (256 + tiles - 1) / tiles;
  if (nz >= 8) nz = (nz + 7) / 8 * 8;
  if (NC == 2) {
    if (k > 5) nz = 80;
    if (nz > nchunk / 4) nz = nchunk / 4 >= 8 ? nchunk / 32 * 8 : nchunk / 4;
  } else if (nz > 128) {
    nz = 128;
  }
  if (nz > nchunk) nz = nchunk;
  if (nz < 1) nz = 1;
  return (int)nz;
}

template <int NC>
static hipError_t launch_group(const RingDwArgs& a, int mg, unsigned blocks, int seg_begin, int seg_end, int add,
                               hipStream_t st) {
  const int nmat = (a.k + 1 - 3 * mg) < 3 ? (a.k + 1 - 3 * mg) : 3;
  if (mg == 0) {
    if (nmat == 3) RING_LAUNCH((ring_dw_direct_kernel<NC, 3, true>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
    else if (nmat == 2) RING_LAUNCH((ring_dw_direct_kernel<NC, 2, true>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
    else RING_LAUNCH((ring_dw_direct_kernel<NC, 1, true>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
  } else {
    if (nmat == 3) RING_LAUNCH((ring_dw_direct_kernel<NC, 3, false>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
    else if (nmat == 2) RING_LAUNCH((ring_dw_direct_kernel<NC, 2, false>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
    else RING_LAUNCH((ring_dw_direct_kernel<NC, 1, false>), dim3(blocks), dim3(256), 0, st, a, mg, seg_begin, seg_end, add);
  }
  return hipGetLastError();
}

// K chunks a workgroup walks per launch, at most.  The workgroups of a K split read the same two operand streams
// and find each other's fragments in their XCD's L2 only while they stay within about 32 chunks of one another
// (4 MiB of L2 against 128 KiB of new operand bytes per chunk step and XCD).  Nothing synchronises them, so over a
// long walk they drift apart and every one fetches its operands from memory for itself: at N = 512, B = 8192 the
// kernel reads 1.02 x its operands over 512 chunks per workgroup, 1.45 x over 2048 and 2.47 x over 8192.  A long
// sequence is therefore cut into segments in time, one launch each (a launch boundary re-aligns the workgroups);
// the launches after the first add to the partial sums.  RINGATTR_DW_SEGMENT overrides the length (0: no cut) and keeps every
// contraction with the kernel that is cut (ring_dw_short_nz).
static int dw_segment_chunks() {
  const char* e = getenv("RINGATTR_DW_SEGMENT");   // read at every call: tests switch it between calls
  return e ? atoi(e) : 640;
}

// Time-step pairs per segment (whole pairs, so that a segment is a contiguous range of chunks).
static long dw_pairs_per_segment(int nbt, int T, int nz) {
  const int npairs = (T + 1) / 2;
  const long nchunk = (long)nbt * npairs;
  const int seg = dw_segment_chunks();
  long pairs_per_seg = npairs;
  if (seg > 0 && nz > 0 && nchunk / nz > seg) {
    pairs_per_seg = ((long)seg * nz) / nbt;
    if (pairs_per_seg < 1) pairs_per_seg = 1;
  }
  return pairs_per_seg;
}

int ring_dw_tiled_segments(int nbt, int T, int nz) {
  const long per = dw_pairs_per_segment(nbt, T, nz);
  return (int)(((T + 1) / 2 + per - 1) / per);
}

// One launch per group of three matrices (a_dim = 2 needs exactly one) and segment.
hipError_t ring_launch_dw_tiled(const RingDwArgs& a, int NC, hipStream_t st) {
  const int NB = 4 * NC / 8;
  const unsigned blocks = (unsigned)(NB * NB * a.nz);
  const int nmg = (a.k + 3) / 3;
  const int npairs = (a.T + 1) / 2;
  const long pairs_per_seg = dw_pairs_per_segment(a.nbt, a.T, a.nz);
  for (int mg = 0; mg < nmg; ++mg) {
    for (long p0 = 0; p0 < npairs; p0 += pairs_per_seg) {
      const long p1 = p0 + pairs_per_seg < npairs ? p0 + pairs_per_seg : npairs;
      const int b = (int)(p0 * a.nbt), e_ = (int)(p1 * a.nbt), add = p0 > 0 ? 1 : 0;
      hipError_t e = hipErrorInvalidValue;
      switch (NC) {
        case 2: e = launch_group<2>(a, mg, blocks, b, e_, add, st); break;
        case 4: e = launch_group<4>(a, mg, blocks, b, e_, add, st); break;
        case 8: e = launch_group<8>(a, mg, blocks, b, e_, add, st); break;
        case 16: e = launch_group<16>(a, mg, blocks, b, e_, add, st); break;
        case 24: e = launch_group<24>(a, mg, blocks, b, e_, add, st); break;
        case 32: e = launch_group<32>(a, mg, blocks, b, e_, add, st); break;
        default: break;
      }
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

// Which of the two kernels contracts: us of either with its reduction, from the chunks a workgroup walks.  A chunk of three matrices
// takes 0.65 us here and 1.13 times that in dw_chunk_waves, where one of two takes hardly less: a wave loads ten fragments a chunk there
// whatever their number.  A launch's start and end take 4 and 5 us a round of 256 workgroups, partial sums are written and read at 5 TB/s.
// Held against 715 shapes, N = 70 to 2048, 1 to 16 channels, 5 to 65536 chunks: the kernel it takes is at most 13 % and 26 us slower
// than the other where it is dw_chunk_waves (N = 200: one channel, 3840 chunks 51 against 45 us, five, 15360 chunks 359 against 340);
// where it stays here some wide rings with many channels would gain from the other (N = 565, seven channels, 43095 chunks 20.8 against
// 15.8 ms; N = 700, 16, 15360 chunks 15.9 against 13.8; most gain nothing).  So long contractions of whole 128 x 128 blocks and those of
// one channel stay here; us, here and there:
//   one channel: N = 512, 15360 chunks 444 and 629, 945 chunks 44 and 42; N = 1024, 3840 chunks 430 and 609; N = 360, 15360 chunks 440
//     and 388
//   two: N = 512, 65536 chunks 2480 and 2810; N = 1024, 3840 chunks 573 and 638; N = 256, 15360 chunks 181 and 214; N = 2048, 160 chunks
//     178 and 194; N = 256, 945 chunks 34 and 25; N = 360 (padded to 512 here), 1890 chunks 87 and 60
//   three (two launches here): N = 256, 15360 chunks 289 and 212
// No launch of dw_chunk_waves is cut in time, however long: the waves of its workgroups drift apart as the others do, and it is ahead all
// the same where it is taken, by the products that padding and a last launch of one matrix cost the other.  us of contraction (GB
// fetched), cut here and there: N = 360, two channels, 131072 chunks 4710 (9.5) and 3290 (10.4), three, 65536 chunks 4280 and 2020;
// N = 640, two, 65536 chunks 10270 and 5570; N = 512, three, 131072 chunks 8630 (18.6) and 7150 (33.7); N = 200, three 2380 and 1560;
// N = 120, six 2970 and 1210.
// Returns the K splits of dw_chunk_waves, 0: not that kernel.
int ring_dw_short_nz(int N, int NC, int k, int nbt, int T, int tiled_nz, int linear_tiles) {
  if (getenv("RINGATTR_DW_SEGMENT")) return 0;             // (asks for the kernel that is cut)
  RingDwArgs a = {};
  a.N = N;
  a.linear_tiles = linear_tiles;
  const int NB = 4 * NC / 8, tiles = dw_tiles(a, 4 * NC), groups = (k + 4) / 4;
  const long nb = (long)((tiles + DW_WI - 1) / DW_WI) * ((tiles + DW_WJ - 1) / DW_WJ), nchunk = (long)nbt * ((T + 1) / 2);
  // as many as fill the chip, each with two chunks a wave at least
  long nz = 256 / nb;
  if (nz > nchunk / 8) nz = nchunk / 8;
  if (nz > tiled_nz) nz = tiled_nz;
  if (nz < 1) nz = 1;
  constexpr float CHUNK = 0.65f, BYTES = 5e6f, tiled_share[4] = {0.f, 0.7f, 0.75f, 1.f}, short_share[5] = {0.f, 0.65f, 1.1f, 1.13f, 1.42f};
  auto chunks = [&](long parts) { return (float)((nchunk + parts - 1) / parts) * CHUNK; };
  const float tiled_rounds = (float)(((long)NB * NB * tiled_nz + 255) / 256), short_rounds = (float)((nb * nz + 255) / 256);
  float tiled = 8.f * tiled_nz * (1 + k) * (64.f * NC) * (64.f * NC) / BYTES, here = 8.f * nz * (1 + k) * (16.f * tiles) * (16.f * tiles) / BYTES;
  for (int m = 0; m <= k; m += 3) tiled += tiled_rounds * (chunks(tiled_nz) * tiled_share[k + 1 - m < 3 ? k + 1 - m : 3] + 4.f);
  for (int m = 0, left = groups; left > 0; --left) {
    const int nm = (k + 1 - m + left - 1) / left;
    here += short_rounds * (chunks(4 * nz) * short_share[nm] + 5.f);
    m += nm;
  }
  return here < tiled ? (int)nz : 0;
}

// Through dw_chunk_waves where that is the faster one; its K splits (no more than there were) go into a.nz.
hipError_t ring_launch_dw_short(RingDwArgs& a, int NC, hipStream_t st) {
  const int nz = ring_dw_short_nz(a.N, NC, a.k, a.nbt, a.T, a.nz, a.linear_tiles);
  if (nz == 0) return ring_launch_dw_tiled(a, NC, st);
  a.nz = nz;
  const int NT = 4 * NC, tiles = dw_tiles(a, NT);
  const int nb = ((tiles + DW_WI - 1) / DW_WI) * ((tiles + DW_WJ - 1) / DW_WJ);
  const dim3 grid((unsigned)(8 * ((nb * nz + 7) / 8)));
  for (int m0 = 0, groups = (a.k + 4) / 4; m0 <= a.k; --groups) {
    const int nm = (a.k + 1 - m0 + groups - 1) / groups;          // matrices shared out evenly
    auto go = [&](auto kern) { RING_LAUNCH(kern, grid, dim3(256), 0, st, a, m0, NT, 0, 0); };
    if (m0 == 0) {
      switch (nm) {
        case 4: go(ring_dw_direct_kernel<0, 4, true>); break;
        case 3: go(ring_dw_direct_kernel<0, 3, true>); break;
        case 2: go(ring_dw_direct_kernel<0, 2, true>); break;
        default: go(ring_dw_direct_kernel<0, 1, true>); break;
      }
    } else {
      switch (nm) {
        case 4: go(ring_dw_direct_kernel<0, 4, false>); break;
        case 3: go(ring_dw_direct_kernel<0, 3, false>); break;
        case 2: go(ring_dw_direct_kernel<0, 2, false>); break;
        default: go(ring_dw_direct_kernel<0, 1, false>); break;
      }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    m0 += nm;
  }
  return hipSuccess;
}
