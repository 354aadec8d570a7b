// Team kernels: choice of shape and scratch area (kernels: ring_team.hpp).
#include "ring_team.hpp"

// Sum of the members' dL/dA partials in member order.
__global__ __launch_bounds__(256) void ring_team_ga_reduce_kernel(const float* __restrict__ part, float* __restrict__ grad_A,
                                                                  int G, int T, int k, int B) {
  const size_t n = (size_t)T * k * B, u = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= n) return;
  float v = 0.f;
  for (int g = 0; g < G; ++g) v += part[(size_t)g * n + u];
  const int b = (int)(u % B);
  const size_t tc = u / B;
  const int ch = (int)(tc % k), t = (int)(tc / k);
  grad_A[((size_t)b * T + t) * k + ch] = v;
}

// The exchange area empty, the teams' words behind it zero.
__global__ __launch_bounds__(256) void ring_team_fill_kernel(u32x4* p, unsigned nx, unsigned n) {
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const unsigned v = i < nx ? EMPTY : 0u;
    p[i] = u32x4{v, v, v, v};
  }
}

#include <stdlib.h>
#include <algorithm>

namespace {

constexpr int XCDS = 8, CUS_PER_XCD = 32;
constexpr size_t LDS_MAX = 160 * 1024;

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

template <int C16, int WK>
size_t plan_lds(const RingTeamShape& s, int k, int nt, int KC, bool bptt, bool ga) {
  return lds_plan<C16, WK>(k, nt, s.lds_mats, KC, parked_bytes(s.kpw, s.c16, s.mr, s.wk), bptt, ga).total;
}

size_t shape_lds(const RingTeamShape& s, int k, int nt, int KC, bool bptt, bool ga) {
  if (s.wk == 4) {
    return s.c16 == 1 ? plan_lds<1, 4>(s, k, nt, KC, bptt, ga)
                      : (s.c16 == 2 ? plan_lds<2, 4>(s, k, nt, KC, bptt, ga) : plan_lds<4, 4>(s, k, nt, KC, bptt, ga));
  }
  return s.c16 == 1 ? plan_lds<1, 8>(s, k, nt, KC, bptt, ga)
                    : (s.c16 == 2 ? plan_lds<2, 8>(s, k, nt, KC, bptt, ga) : plan_lds<4, 8>(s, k, nt, KC, bptt, ga));
}

const RingTeamShape kShapes[] = {
#define RING_TEAM_ROW(KPW, C16, MR, WK, FEW, MORE) {KPW, C16, MR, WK, MORE ? TEAM_MORE : FEW, 0},      // (lds_mats here: how many there may be)
    RING_TEAM_SHAPES(RING_TEAM_ROW)
#undef RING_TEAM_ROW
};

int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return cus;
}

}  // namespace

// The shape of a team for this problem: the cheapest of the built ones by a model of one time step in cycles.
//   products of an item  M c16 KC 16 / 4 (four matrix pipes) + reading the fragments kept in LDS + what a wave spends around them
//   epilogue of an item  grows with the outputs per auxiliary thread
//   one tile per team:   products + epilogue + hand-over through L2, one after the other
//   more tiles:          products and epilogue of neighbouring items overlap
RingTeamPlan ring_team_plan(int N, int k, int T, int B, bool bptt, bool ga) {
  RingTeamPlan best{};
  best.ok = false;
  if (N < 17 || N > 1024 || k < 1 || k > 16 || T < 1 || B < 1) return best;
  const int KC = (N + 31) / 32, nbt = (B + 15) / 16;
  for (const RingTeamShape& s0 : kShapes) {
    RingTeamShape s = s0;
    if (s.wk == 4 ? KC > 4 : KC <= 4) continue;
    if (s.kpw != (KC + s.wk - 1) / s.wk) continue;
    s.lds_mats = std::max(0, k + 1 - s.mr);
    if (s.lds_mats > s0.lds_mats) continue;
    const int G = (2 * KC + s.c16 - 1) / s.c16;
    if (G > CUS_PER_XCD) continue;
    const int nteams = std::min(nbt, XCDS * (CUS_PER_XCD / G)), nt = (nbt + nteams - 1) / nteams;
    const int slots = nt == 1 ? 8 : (nt < 4 ? 6 : 4);
    const size_t xbytes = (size_t)slots * nbt * KC * CHUNK_BYTES;
    if (xbytes >= ((size_t)1 << 30)) continue;     // (offsets past the buffer say 'nowhere')
    if (shape_lds(s, k, nt, KC, bptt, ga) > LDS_MAX) continue;
    s.grid = XCDS * G * ((nteams + XCDS - 1) / XCDS);
    const float npt = s.c16 == 4 ? 4.f : 2.f;
    const float prod = 4.4f * (float)(std::max(s.mr, k + 1) * s.c16 * s.kpw * s.wk) + 4.f * (float)(s.lds_mats * s.c16 * KC) + 250.f;
    const float epi = 350.f + 110.f * npt;
    const float one = prod + epi + 650.f;
    const float step = nt == 1 ? one : std::max(one, (float)nt * (std::max(prod, epi) + 60.f));
    if (!best.ok || step < best.step_cycles) {
      best.ok = true;
      best.shape = s;
      best.KC = KC;
      best.G = G;
      best.nteams = nteams;
      best.nt = nt;
      best.slots = slots;
      best.xchg_bytes = up256(xbytes);
      best.gather_bytes = (size_t)nteams * RING_TEAM_WORD * sizeof(unsigned long long);
      best.ga_bytes = ga ? up256((size_t)G * T * k * B * sizeof(float)) : 0;
      best.step_cycles = step;
    }
  }
  return best;
}

static bool forced() {
  const char* v = getenv("RINGATTR_TEAM");
  return v && v[0] == '1';
}

// Whether a workgroup per 4 to 16 rows does it; RINGATTR_TEAM=1 asks for the exchange through L2.
bool ring_uses_team_one(int N, int k) { return ring_team_one_applicable(N, k) && !forced(); }

// Where teams run (us per time step, measured with T = 60, gelu; forward for inference / forward + backward):
//   N = 360, a_dim 2:  B = 64: 8.2 -> 1.5 / 30.6 -> 3.4   B = 1024: 12.9 -> 3.3 / 31.9 -> 7.8   B = 4096: 15.6 -> 8.0 / 37 -> 23
//   N = 512, a_dim 2:  B = 64: 8.9 -> 1.6 / 29.1 -> 3.7   B = 2048: 14.3 -> 5.5 / 32.4 -> 14.8
//   N = 1024, a_dim 2: B = 64: 17.8 -> 3.3 / 43 -> 6.9    B = 2048: 40 -> 19 / 104 -> 50
// against the streaming and step-per-launch kernels.  The exceptions:
//   * up to 128 neurons and six channels a workgroup holds the whole ring (ring_team_one.hip); more channels run on teams
//     (N = 120, a_dim 2, B = 64, while it ran on teams of eight: 2.5 -> 0.9 / 5.8 -> 2.3);
//   * 128 < N <= 256 with two channels belongs to the weight-resident kernels, which are far ahead on large batches (N = 200,
//     B = 4096, forward and backward: 7.4 against 10.5).  A slice of a batch has to reproduce its rows bit for bit and the two
//     families sum in a different order, so batches of up to 512 rows run on teams that sum in the weight-resident order
//     (ring_team_rows.hip; N = 200, B = 64: 2.0 against 3.8 on the weight-resident kernels and 3.0 on these teams);
//   * with many tiles per team (more than eight at N <= 512) a compute unit's epilogue work is what bounds a step, and
//     the kernels that have a batch tile to themselves, or the N = 512 clusters, are faster (N = 360, B = 6000, forward
//     and backward: 49 against 43 us per step with nine tiles, B = 8192: 53 against 68 with thirteen; N = 512, B = 4608:
//     46 against 37, B = 6016: 49 against 54).  Rows reproduce between batches on the same side of this line: members of
//     any width sum a row alike.
// The rule does not ask whether a record is wanted: a history is the same with and without one.
static bool team_shape(int N, int k, int T, int B) {
  if (ring_uses_team_one(N, k)) return true;
  if (ring_res256_applicable(N, k) && !forced()) return false;
  const RingTeamPlan f = ring_team_plan(N, k, T, B, false, false);
  if (!f.ok || !ring_team_plan(N, k, T, B, true, true).ok) return false;
  return forced() || N > 512 || f.nt <= 8;
}

bool ring_teams_allowed() {
  const char* v = getenv("RINGATTR_TEAM");
  if ((v && v[0] == '0') || ring_cluster_error()) return false;
  // a switch that asks for one of the other families by name is obeyed
  for (const char* name : {"RINGATTR_STREAMING", "RINGATTR_ROW_TILES", "RINGATTR_BLOCK", "RINGATTR_WIDE", "RINGATTR_SPLIT_FORWARD",
                           "RINGATTR_LDS_WEIGHTS", "RINGATTR_BLOCK_SHAPE", "RINGATTR_CLUSTER", "RINGATTR_CLUSTER_BPTT"})
    if (getenv(name)) return false;
  return device_cus() == XCDS * CUS_PER_XCD;
}

bool ring_uses_team(int N, int k, int T, int B) { return ring_teams_allowed() && team_shape(N, k, T, B); }

// Same bits and record as the weight-resident kernels, so the batch may decide: wherever every batch tile gets a team.
bool ring_uses_team_rows(int N, int k, int B, bool record) {
  return !forced() && ring_teams_allowed() && ring_uses_resident(N, k) && ring_team_rows_plan(N, k, B, record).ok;
}
size_t ring_team_rows_bytes(int N, int k, int B, bool record) {
  const RingTeamPlan p = ring_team_rows_plan(N, k, B, record);
  return p.ok ? p.xchg_bytes + p.gather_bytes : 0;
}
size_t ring_team_rows_bptt_bytes(int N, int k, int T, int B, bool ga) {
  return ring_team_rows_bytes(N, k, B, true) + (ga ? ring_team_rows_ga_bytes(T, B) : 0);
}

// Scratch of one launch; none where no call of this shape comes here.
static size_t plan_bytes(int N, int k, int T, int B, bool bptt, bool ga) {
  if (!team_shape(N, k, T, B) || ring_uses_team_one(N, k)) return 0;
  const RingTeamPlan p = ring_team_plan(N, k, T, B, bptt, ga);
  return p.xchg_bytes + p.gather_bytes + p.ga_bytes;
}
size_t ring_team_fwd_bytes(int N, int k, int T, int B) { return plan_bytes(N, k, T, B, false, false); }
size_t ring_team_bptt_bytes(int N, int k, int T, int B, bool ga) { return plan_bytes(N, k, T, B, true, ga); }

// How long a wait inside the time loop polls, and how long members wait for each other before it (RingTeamArgs).
void ring_team_limits(int* spin_max, int* gather_ticks) {
  *spin_max = 16000000;   // some seconds of polling
  if (const char* v = getenv("RINGATTR_CLUSTER_SPIN")) {
    const long s = atol(v);
    if (s >= -1 && s <= 100000000L) *spin_max = (int)s;
  }
  // A team whose compute units are busy waits about as long as the way round it takes (some 50 ms at N = 1024, T = 120).
  *gather_ticks = 5000000;
  if (const char* v = getenv("RINGATTR_TEAM_GATHER_US")) {
    const long us = atol(v);
    if (us >= -1 && us <= 10000000L) *gather_ticks = us < 0 ? -1 : (int)us * 100;
  }
}

hipError_t ring_team_fill(void* ws, size_t xchg_bytes, size_t gather_bytes, hipStream_t st) {
  const unsigned nx = (unsigned)(xchg_bytes / 16), n = (unsigned)((xchg_bytes + gather_bytes) / 16);
  hipLaunchKernelGGL(ring_team_fill_kernel, dim3(std::min(1024u, (n + 255) / 256)), dim3(256), 0, st, reinterpret_cast<u32x4*>(ws), nx, n);
  return hipGetLastError();
}

// RingTeamArgs::look (measured: team_look).
static int first_look(const RingTeamPlan& p, bool bptt) {
  if (p.nt != 1 || !team_may_look_late(p.shape.kpw, p.shape.c16, p.shape.mr, p.shape.wk, p.shape.lds_mats)) return -1;
  return p.shape.kpw < 3 ? 8 : bptt ? 10 : 12;
}

static hipError_t team_args(const RingTeamPlan& p, const float* Wo, const float* Wa, const float* A, float J0, float J1,
                            bool folded, int N, int k, int T, int B, int cts, int look, void* ws, RingTeamArgs& c,
                            hipStream_t st) {
  hipError_t e = ring_cluster_host_err(&c.host_err);
  if (e != hipSuccess) return e;
  c.xchg = ws;
  c.xchg_bytes = (unsigned)p.xchg_bytes;
  c.Wo = Wo;
  c.Wa = Wa;
  c.A = A;
  c.gather = reinterpret_cast<unsigned long long*>(static_cast<char*>(ws) + p.xchg_bytes);
  c.ga_part = reinterpret_cast<float*>(static_cast<char*>(ws) + p.xchg_bytes + p.gather_bytes);
  c.scale0 = folded ? J1 : 1.f;
  c.shift0 = folded ? J0 : 0.f;
  c.J0 = folded ? 0.f : J0;
  c.J1 = folded ? 1.f : J1;
  c.N = N;
  c.k = k;
  c.T = T;
  c.B = B;
  c.nbt = (B + 15) / 16;
  c.KC = p.KC;
  c.G = p.G;
  c.nteams = p.nteams;
  c.nt = p.nt;
  c.slots = p.slots;
  c.cts = cts;
  ring_team_limits(&c.spin_max, &c.gather_ticks);
  c.c16 = p.shape.c16;
  c.mr = p.shape.mr;
  c.wk = p.shape.wk;
  c.rows = 0;
  c.look = look;
  return ring_team_fill(ws, p.xchg_bytes, p.gather_bytes, st);
}

// (the fields that a workgroup on its own needs)
static RingTeamArgs one_args(const float* Wo, const float* Wa, const float* A, float J0, float J1, int N, int k, int T, int B, int cts) {
  RingTeamArgs c = {};
  c.Wo = Wo;
  c.Wa = Wa;
  c.A = A;
  c.J0 = J0;
  c.J1 = J1;
  c.N = N;
  c.k = k;
  c.T = T;
  c.B = B;
  c.cts = cts;
  return c;
}

hipError_t ring_team_fwd(const RingFwdArgs& a, const float* Wo, const float* Wa, bool folded, int cts, void* ws, hipStream_t st) {
  if (ring_uses_team_one(a.N, a.k)) return ring_launch_team_one_fwd(a, one_args(Wo, Wa, a.A, a.J0, a.J1, a.N, a.k, a.T, a.B, cts), st);
  const RingTeamPlan p = ring_team_plan(a.N, a.k, a.T, a.B, false, false);
  if (!p.ok || !ws || (a.dfrag != nullptr) != (a.rfrag != nullptr)) return hipErrorInvalidValue;
  RingTeamArgs c;
  hipError_t e = team_args(p, Wo, Wa, a.A, a.J0, a.J1, folded, a.N, a.k, a.T, a.B, cts, first_look(p, false), ws, c, st);
  if (e != hipSuccess) return e;
  e = ring_launch_team_fwd(a, c, p.shape, st);
  return e == hipSuccess ? ring_launch_team_solo_fwd(a, c, st) : e;
}

// The split that leaves room for the launches of other streams that have not finished; under capture for one beside this one.
static RingTeamPlan rows_plan_on(hipStream_t st, int N, int k, int B, bool record) {
  const int others = ring_launch_guard().beside(st);
  return ring_team_rows_plan(N, k, B, record, others < 0 ? 2 : others + 1);
}

hipError_t ring_team_rows(const RingFwdArgs& a, const float* Wo, const float* Wa, void* ws, hipStream_t st) {
  const bool record = a.dfrag != nullptr;
  const RingTeamPlan p = rows_plan_on(st, a.N, a.k, a.B, record);
  if (!p.ok || !ws || !a.hist || record != (a.rfrag != nullptr)) return hipErrorInvalidValue;
  RingTeamArgs c;
  hipError_t e = team_args(p, Wo, Wa, a.A, a.J0, a.J1, true, a.N, a.k, a.T, a.B, 16, a.B <= 8 ? 8 : 10, ws, c, st);
  if (e != hipSuccess) return e;
  c.wk = 1;
  c.rows = a.N == 256 && a.B % 16 == 0 ? 2 : 1;
  e = ring_launch_team_rows(a, c, p.shape, st);
  if (e == hipSuccess) e = ring_launch_team_solo_fwd(a, c, st);
  return e == hipSuccess && a.loss_stats ? ring_launch_row_sums256(a.hist, a.loss_stats, a.N, a.T, a.B, st) : e;
}

hipError_t ring_team_rows_bptt(const RingBpttArgs& a, const float* Wo, const float* Wa, void* ws, hipStream_t st) {
  const RingTeamPlan p = rows_plan_on(st, a.N, a.k, a.B, true);
  if (!p.ok || !ws) return hipErrorInvalidValue;
  RingTeamArgs c;
  hipError_t e = team_args(p, Wo, Wa, a.A, a.J0, a.J1, true, a.N, a.k, a.T, a.B, 16, 8, ws, c, st);
  if (e != hipSuccess) return e;
  c.wk = c.rows = 1;
  e = ring_launch_team_rows_bptt(a, c, p.shape, st);
  if (e == hipSuccess) e = ring_launch_team_solo_bptt(a, c, st);
  return e == hipSuccess && a.grad_A ? ring_launch_team_rows_ga(c.ga_part, a.grad_A, a.T, a.B, st) : e;
}

hipError_t ring_team_rebuild(const RingFwdArgs& a, bool folded, int cts, hipStream_t st) {
  const bool one = ring_uses_team_one(a.N, a.k);           // (sums in the order of a single compute wave)
  const RingTeamPlan p = one ? RingTeamPlan{} : ring_team_plan(a.N, a.k, a.T, a.B, false, false);
  if (!one && !p.ok) return hipErrorInvalidValue;
  RingTeamArgs c = {};
  c.A = a.A;
  c.J0 = folded ? 0.f : a.J0;
  c.J1 = folded ? 1.f : a.J1;
  c.k = a.k;
  c.KC = (a.N + 31) / 32;
  c.cts = cts;
  return ring_launch_team_rebuild(a, c, one ? 1 : p.shape.wk, st);
}

hipError_t ring_team_bptt(const RingBpttArgs& a, const float* Wo, const float* Wa, bool folded, int cts, void* ws, hipStream_t st) {
  const bool ga = a.grad_A != nullptr;
  if (ring_uses_team_one(a.N, a.k)) return ring_launch_team_one_bptt(a, one_args(Wo, Wa, a.A, a.J0, a.J1, a.N, a.k, a.T, a.B, cts), st);
  const RingTeamPlan p = ring_team_plan(a.N, a.k, a.T, a.B, true, ga);
  if (!p.ok || !ws) return hipErrorInvalidValue;
  RingTeamArgs c;
  hipError_t e = team_args(p, Wo, Wa, a.A, a.J0, a.J1, folded, a.N, a.k, a.T, a.B, cts, first_look(p, true), ws, c, st);
  if (e != hipSuccess) return e;
  e = ga ? ring_launch_team_bptt_ga(a, c, p.shape, st) : ring_launch_team_bptt(a, c, p.shape, st);
  if (e == hipSuccess) e = ring_launch_team_solo_bptt(a, c, st);
  if (e != hipSuccess || !ga) return e;
  const size_t n = (size_t)a.T * a.k * a.B;
  hipLaunchKernelGGL(ring_team_ga_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, c.ga_part, a.grad_A, p.G, a.T, a.k, a.B);
  return hipGetLastError();
}
