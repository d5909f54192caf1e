// flow.hip -- continuous-batching server of O(N) LPA flows with an on-device RK4 stepper.
//
// Each flow evolves u(rho) = U'(rho) on a uniform rho grid from k = Lambda = 1 to k_end with fixed
// RK4 steps in t = ln(Lambda/k):
//   du/dt = 1/2 [ (N-1) u' I_T(u) + (3 u' + 2 rho u'') I_T(u + 2 rho u') ],
//   I_T(m2) = int d^3q/(2pi)^3 RBdot(k^2,q^2) S2(E),  E^2 = q^2 + RB(k^2,q^2) + m2,
//   S2(E) = T sum_n (w_n^2 + E^2)^-2 = coth(E/2T)/(4E^3) + csch^2(E/2T)/(8 T E^2),
// i.e. two threshold integrals (the d = 3 radial form of IntegratorGPU<3>, integrator_gpu.hh:34-60,
// with the closed-form bosonic Matsubara sum, cf. Examples/ONfiniteT/flows/V/V.kernel) per grid
// point and RK stage.  u', u'' are second-order finite differences (one-sided at the ends).
//
// Device layout: every resident flow owns 2 n doubles in one HBM pool (u after even and after odd
// steps).  The host cuts the resident flows into runs of consecutive grid points; one launch
// advances every run by a whole RK4 step, one workgroup per run, evaluating the stages outside the
// run as far as the next stages' stencils reach (flow_step_kernel).  steps_per_launch steps are
// captured into one hipGraph.  A flow's step index is the launch's base step plus the step within
// the graph minus the base step at its admission, so flows admitted at different times share the
// graph and a finished flow simply stops updating.  The graph's last node advances the device copy
// of the base step, which the host mirrors.  Between graph launches the host retires finished and
// non-finite flows and admits queued ones while their HBM footprint fits the budget.
//
// Node factors: with x_j the GL nodes, xr_j = x_j x_extent, the regulator terms are
// q^2 = k^2 xr, R = k^2 e^-xr, RBdot = 2 k^2 e^-xr (1 + xr) and the d = 3 element times weight is
// k^3 sqrt(xr) w_j x_extent / (4 pi^2), so per node only A_j = xr_j + e^-xr_j (E^2 = k^2 A_j + m^2)
// and D_j = sqrt(xr_j) w_j x_extent e^-xr_j (1 + xr_j) / (2 pi^2) (element * weight * RBdot = k^5 D_j)
// depend on j; both are fixed by the quadrature and tabulated once.  k(t) is tabulated per step and
// stage exactly as the oracle's stepper forms it.
#include "internal.hh"
#include "dfrg/device.hh"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <cmath>
#include <deque>
#include <map>
#include <vector>

using namespace dfrg;

namespace
{
  constexpr double kPi = 3.14159265358979323846;
  constexpr double kLog2e = 1.4426950408889634074;

  // A run of consecutive grid points [a, b) of one resident flow, which one workgroup advances by
  // a whole RK4 step, with the flow's parameters (one record per run, so a step's loads depend on
  // it alone).  Runs are at least 2 points long (the one-sided stencils at the grid ends then find
  // their points in the previous stage's range).
  struct FlowRun {
    int slot, a, b, n, off, admit;
    double h, i2h, ih2; // grid spacing, 1/(2 h), 1/h^2
    double T, N;        // temperature, O(N)
    double m2_0, lam;   // initial condition u(rho) = m2_0 + lam/2 rho (step 0 starts from it)
  };

  constexpr int kRunBlock = 1024;                 // threads per workgroup: 16 waves share a run
  constexpr int kHalo = 3;                        // stages 1-3 are also evaluated this far outside the run
  constexpr int kMaxRun = 250;                    // longest run
  constexpr int kSpan = kMaxRun + 2 * (kHalo + 1); // the run and the stencil reach of its stage 1
  // run lengths whose first stage (6 points more) fills whole waves on the four SIMDs
  constexpr int kRunLengths[] = {2, 6, 10, 18, 26, 42, 58, 74, 90, 106, 122, 154, 186, 218, 250};
  constexpr int kMaxFlowGrid = 1024;              // most workgroups of a step launch, grid-stride over runs
  constexpr int kFlowGraphs = 5;                  // step graphs, with grids of 64, 128, ... kMaxFlowGrid
  static_assert(64 << (kFlowGraphs - 1) == kMaxFlowGrid);

  struct FlowDev {
    int *bad;             // per slot: a non-finite value appeared
    FlowRun *runs;        // every resident flow cut into runs
    int *n_runs;          // device copy of the run count
    int *base;            // global step index of the first step of this launch
    double *pool;         // state: u at even steps | u at odd steps, per flow
    const double2 *nodes; // node factors (A_j, D_j/4) (header comment), padded to a multiple of 64 with
                          // (1e30, 0), whose terms are zeros
    const double *exp2t;  // 2^(j/512), j = 0..511
    const double *kt;     // k at (step, stage point): 3 per step, t, t + dt/2, t + dt
    int nx, n_steps;
    double dt;
  };
  // 2^(a b/512) for |a b| < 2^30: exp2t[j] = 2^(j/512), dev::exp2_tab's rounding, and 2^(f/512) - 1 =
  // f P(f) with P of degree 3 (remainder 1.3e-19).
  constexpr int kFlowExp = 512;
  __device__ __forceinline__ double exp2_tab512(double a, double b, const double *exp2t)
  {
    constexpr double kRound = 6755399441055744.0;
    const double sh = fma(a, b, kRound);
    const int jn = __double2loint(sh);
    const double f = fma(a, b, -(sh - kRound));
    double p = fma(f, 1.399622015673666e-13, 4.1353784454173436e-10);
    p = fma(p, f, 9.163913992275265e-07);
    p = fma(p, f, 0.001353803087031143);
    const double c = exp2t[jn & (kFlowExp - 1)];
    return ldexp(fma(c * f, p, c), jn >> 9);
  }

  // The temperature's factors in bose_4S2.
  struct Bose {
    double two_inv_T, exp_scale, E_max; // 2/T, -512 log2(e)/T, 1000 T
    __device__ __forceinline__ explicit Bose(double T)
    {
      const double inv_T = 1.0 / T;
      two_inv_T = 2.0 * inv_T;
      exp_scale = -512.0 * kLog2e * inv_T;
      E_max = 1000.0 * T;
    }
  };
  // 4 S2(E) with S2 = coth(E/2T)/(4E^3) + csch^2(E/2T)/(8 T E^2), e = exp(-E/T), coth = (1+e)/(1-e),
  // csch^2 = 4e/(1-e)^2, r = 1/(1-e) and y = 1/E:
  //   4 S2 = y^3 r^2 (1 - e^2 + 2 (E/T) e),
  // by FP64 forms instead of library calls: y and r from FP32 hardware seeds and one Newton step, e by
  // table (E/T beyond 1000 gives 0 through the exponent).  1 - e loses relative accuracy only as
  // E/T -> 0 (absolute error ~1e-16 against 1 - e ~ E/T).  Relative error ~1e-14.  E2 <= 0 gives NaN.
  // 38 VALU instructions against 47 with the temperature's factors inside and a 64-entry table.  (FP64
  // seeds would take 32, but a flow can carry the 1e-14 they differ by to 3e-11 in its final u.)
  __device__ __forceinline__ double bose_4S2(double E2, const Bose &B, const double *exp2t)
  {
    const double y = dev::rsqrt_seeded(E2);
    const double E = fmin(E2 * y, B.E_max);
    const double e = exp2_tab512(E, B.exp_scale, exp2t);
    const double r = dev::rcp_seeded(1.0 - e);
    const double q = fma(B.two_inv_T, E * e, fma(-e, e, 1.0));
    return (y * y * y) * (r * r) * q;
  }

  // a + b with no product fused into it
  __device__ __forceinline__ double add_plain(double a, double b)
  {
#pragma clang fp contract(off)
    return a + b;
  }

  // The lanes of one grid point: NL lanes for the threshold integral at u (kind 0), the next NL for
  // the one at u + 2 rho u' (kind 1); a lane sums 64/NL nodes of each chunk of 64.
  // Node sums are one tree over the bits of the node index, 5, 4, 3 (in the lane or across lanes,
  // by NL), then 0, 1, 2 across eight lanes, so a sum's bits do not depend on NL.
  template <int NL> __device__ __forceinline__ double node_tree(double (&t)[NL == 32 ? 2 : 4])
  {
#pragma clang fp contract(off) // a product fused into its first addition would depend on NL
#pragma unroll
    for (int s = NL == 32 ? 1 : 2; s >= 1; s >>= 1)
#pragma unroll
      for (int i = 0; i < s; ++i) t[i] += t[i + s];
    double v = t[0];
    if constexpr (NL == 32) v = dev::pair_sum16(v, v); // bit 4
    if constexpr (NL >= 16) v += dev::dpp_f64<0x128>(v); // bit 3
    v += dev::dpp_f64<0xB1>(v);
    v += dev::dpp_f64<0x4E>(v);
    v += dev::dpp_f64<0x141>(v);
    return v;
  }
  // The sums of kind 0 and kind 1 of this lane's point, to all its lanes.
  template <int NL> __device__ __forceinline__ void both_kinds(double v, int kind, double &i0, double &i1)
  {
    if constexpr (NL == 8) {
      const double o = dev::dpp_f64<0x128>(v); // the other eight lanes of the row
      i0 = kind ? o : v;
      i1 = kind ? v : o;
    } else {
      dev::swap_halves<NL>(v, i0, i1);
    }
  }

  // The four stages of one run.  x0: grid point of LDS entry 0; entry p belongs to slot (p - 1) mod SLOTS.
  template <int NL>
  __device__ __forceinline__ void flow_stages(const FlowDev &F, const FlowRun &run, int step, double *u_new,
                                              const double2 *s_nodes, const double *s_exp2, double *s_u,
                                              double *s_acc, double (*s_y)[kSpan])
  {
    constexpr int SLOTS = kRunBlock / (2 * NL), EV = 64 / NL, UN = EV < 4 ? EV : 4;
    const int tid = threadIdx.x, sub = tid & (NL - 1), kind = (tid / NL) & 1, slot = tid / (2 * NL);
    const int n = run.n, a = run.a, b = run.b, x0 = a - kHalo - 1;
    const double dt = F.dt;
    const Bose B(run.T);
    const double k_t = F.kt[3 * step], k_half = F.kt[3 * step + 1], k_dt = F.kt[3 * step + 2];
    // up to four nodes per lane stay in registers
    constexpr bool KEEP = EV <= 4;
    double2 kept[KEEP ? EV : 1];
    if (KEEP)
#pragma unroll
      for (int i = 0; i < (KEEP ? EV : 1); ++i) kept[i] = s_nodes[sub + NL * i];
    for (int stage = 1; stage <= 4; ++stage) {
      const int w = 4 - stage;
      const int p0 = max(a - w, 0) - x0, p1 = min(b + w, n) - x0; // evaluated entries [p0, p1)
      const double k = stage == 1 ? k_t : (stage == 4 ? k_dt : k_half);
      const double k2 = k * k, k5 = k2 * k2 * k;
      const double *y = stage == 1 ? s_u : s_y[stage & 1];
      double *y_next = s_y[(stage & 1) ^ 1];
      for (int p = 1 + slot; p < p1; p += SLOTS) {
        if (p < p0) continue;
        // second-order stencils; at a grid end the neighbours of the next point inside, with the
        // one-sided first derivative (d -+ 2 dd)/(2h)
        const int x = x0 + p, in = x == 0 ? 1 : x == n - 1 ? -1 : 0;
        const double yv = y[p], yl = y[p + in - 1], yc = y[p + in], yr = y[p + in + 1];
        const double dd = (yr - 2.0 * yc) + yl;
        const double up = fma(-2.0 * in, dd, yr - yl) * run.i2h, upp = dd * run.ih2;
        const double rho2 = 2.0 * (x * run.h);
        const double m2 = kind ? fma(rho2, up, yv) : yv;
        double v = 0.0;
        for (int c = 0; c < F.nx; c += 64) {
          // four nodes at a time; the second four of NL = 8 add bit 5
          double t[UN];
#pragma unroll 1
          for (int g = 0; g < EV; g += UN)
#pragma unroll
            for (int i = 0; i < UN; ++i) {
              const double2 nd = KEEP && c == 0 ? kept[KEEP ? i : 0] : s_nodes[c + sub + NL * (g + i)];
              const double e = nd.y * bose_4S2(fma(k2, nd.x, m2), B, s_exp2);
              t[i] = g == 0 ? e : add_plain(t[i], e);
            }
          v += node_tree<NL>(t);
        }
        double i0, i1;
        both_kinds<NL>(v, kind, i0, i1);
        const double f = 0.5 * k5 * ((run.N - 1.0) * up * i0 + (3.0 * up + rho2 * upp) * i1);
        // the RK4 stage update, by the point's first lane
        if (kind == 0 && sub == 0) {
          const double u = s_u[p];
          if (stage == 1) {
            s_acc[p] = f;
            y_next[p] = u + 0.5 * dt * f;
          } else if (stage < 4) {
            s_acc[p] += 2.0 * f;
            y_next[p] = u + (stage == 2 ? 0.5 * dt : dt) * f;
          } else {
            const double un = u + dt / 6.0 * (s_acc[p] + f);
            u_new[x] = un;
            if (!isfinite(un)) atomicOr(&F.bad[run.slot], 1);
          }
        }
      }
      __syncthreads();
    }
  }

  // One RK4 step of every resident flow.  A workgroup takes a run [a, b) of one flow and keeps the
  // flow's values at the points [a - kHalo - 1, b + kHalo] in LDS.  Stage s (halo w = 4 - s)
  // evaluates the right-hand side at the points of [a - w, b + w) inside the grid, from the
  // previous stage's values at their neighbours, which the previous stage computed on a range one
  // point wider: points outside the run are evaluated again by the workgroup that owns them, with
  // the same inputs and arithmetic, so every point's result is what a stage-by-stage sweep gives
  // and does not depend on how flows are cut into runs.  u is read from the buffer of this step's
  // parity and written to the other, so neighbouring runs read the old u.
  //
  // What bounds it: VALU issue when the runs fill the CUs, the dependent chain of a stage (stencil,
  // nodes, reduction, update, barrier) when they do not.  So a point's two integrals sit in
  // neighbouring lanes that also form its stencil and its update (one barrier per stage, no hand-over
  // through LDS but the stage's value), eight lanes each, so that a lane has eight independent nodes in
  // flight and the reduction is three steps; short runs spread a point over 16 or 32 lanes.  With a
  // node per lane, 64-lane reductions and three barriers a step of 13,054 points took 22.2 us, of one
  // 64-point flow 9.4; now 16.7 and 6.2.
  __global__ __launch_bounds__(kRunBlock, 4) void flow_step_kernel(FlowDev F, int local)
  {
    extern __shared__ double2 s_nodes[]; // F.nodes
    __shared__ double s_exp2[kFlowExp];
    __shared__ double s_u[kSpan], s_acc[kSpan], s_y[2][kSpan];
    const int tid = threadIdx.x;
    const int R = *F.n_runs, base = *F.base + local;
    // the first run's record is loaded beside the count (the table has kMaxFlowGrid entries at least)
    if (F.runs[blockIdx.x].n == 0 || (int)blockIdx.x >= R) return;
    for (int j = tid; j < (F.nx + 63) / 64 * 64; j += kRunBlock) s_nodes[j] = F.nodes[j];
    for (int j = tid; j < kFlowExp; j += kRunBlock) s_exp2[j] = F.exp2t[j];
    for (int r = blockIdx.x; r < R; r += gridDim.x) {
      const FlowRun run = F.runs[r]; // workgroup-uniform
      const int step = base - run.admit;
      if (step < 0 || step >= F.n_steps) continue; // outside its steps (workgroup-uniform)
      const int n = run.n, len = run.b - run.a, x0 = run.a - kHalo - 1;
      const double *u_old = F.pool + run.off + (step & 1) * n;
      double *u_new = F.pool + run.off + ((step + 1) & 1) * n;
      // step 0 starts from the initial condition itself, so admission copies nothing to the device
      for (int i = tid; i < len + 2 * (kHalo + 1); i += kRunBlock) {
        const int x = x0 + i;
        s_u[i] = x >= 0 && x < n ? (step == 0 ? run.m2_0 + 0.5 * run.lam * (x * run.h) : u_old[x]) : 0.0;
      }
      __syncthreads();
      if (len + 2 * kHalo <= kRunBlock / 64) // 16 points
        flow_stages<32>(F, run, step, u_new, s_nodes, s_exp2, s_u, s_acc, s_y);
      else if (len + 2 * kHalo <= kRunBlock / 32)
        flow_stages<16>(F, run, step, u_new, s_nodes, s_exp2, s_u, s_acc, s_y);
      else
        flow_stages<8>(F, run, step, u_new, s_nodes, s_exp2, s_u, s_acc, s_y);
    }
  }

  // last node of each graph launch: the next launch starts spl steps later
  __global__ void flow_base_kernel(int *base, int spl)
  {
    if (threadIdx.x == 0) *base += spl;
  }

  double now_s()
  {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
  }
} // namespace

struct FlowRecord {
  dfrg_flow_desc desc;
  int state = 0; // 0 queued, 1 resident, 2 finished, 3 failed
  double t_submit = 0, t_done = 0;
  int slot = -1, off = -1, admit = 0;
  std::vector<double> u;
};

// The per-slot flags and the run count live in one device block with a pinned host mirror: the
// host edits the mirror and uploads it with one asynchronous copy before a launch, and the
// launch's non-finite flags come back into the mirror behind the graph.
struct SlotLayout {
  size_t n_runs = 0, bad = 0, bytes = 0;
};

struct dfrg_fs {
  size_t budget = 0;
  int max_resident = 0, nx = 64, n_steps = 2000, steps_per_launch = 10;
  double k_end = 1e-3, x_extent = 20.0;
  FlowDev dev{};
  size_t pool_doubles = 0;
  std::vector<std::pair<int, int>> free_ranges; // (offset, length) in doubles, sorted by offset
  std::vector<long long> slot_flow;             // flow id per slot, -1 idle
  std::map<long long, FlowRecord> flows;
  std::deque<long long> queue;
  long long next_id = 1;
  bool runs_dirty = true;
  size_t runs_cap = 0; // FlowRun entries allocated on the device
  hipStream_t stream = nullptr;
  hipGraph_t graph[kFlowGraphs] = {};
  hipGraphExec_t graph_exec[kFlowGraphs] = {};
  int base = 0;           // global step index of the next launch's first step (mirrors dev.base)
  double *d_nodes = nullptr; // (A, D/4) | 2^(j/512) | kt
  std::vector<double> latencies;
  double busy_s = 0;
  int finished = 0;
  // graph launches: HIP events around each on the server's stream, their summed device time, and
  // the grid-point RK4 steps they advanced
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  long long launches = 0, point_steps = 0;
  double device_s = 0;
  // slot block (device) and its pinned mirror; pinned staging of the run table and of the final u
  // of the flows that end in a launch (copied back behind the graph)
  SlotLayout sl;
  char *d_slots = nullptr, *h_slots = nullptr;
  bool slots_dirty = true;
  FlowRun *h_runs = nullptr;
  size_t h_runs_cap = 0;
  int runs_upload = 0;
  double *h_u = nullptr;
  size_t h_u_cap = 0;
  std::vector<std::pair<int, size_t>> u_staged; // (slot, offset in h_u) of this launch's finishers
  template <class T> T *mirror(size_t off) { return (T *)(h_slots + off); }
};

namespace
{
  int fs_alloc_range(dfrg_fs *fs, int len)
  {
    for (size_t r = 0; r < fs->free_ranges.size(); ++r) {
      auto &fr = fs->free_ranges[r];
      if (fr.second >= len) {
        const int off = fr.first;
        fr.first += len;
        fr.second -= len;
        if (fr.second == 0) fs->free_ranges.erase(fs->free_ranges.begin() + r);
        return off;
      }
    }
    return -1;
  }

  void fs_free_range(dfrg_fs *fs, int off, int len)
  {
    fs->free_ranges.push_back({off, len});
    std::sort(fs->free_ranges.begin(), fs->free_ranges.end());
    std::vector<std::pair<int, int>> merged;
    for (auto &r : fs->free_ranges) {
      if (!merged.empty() && merged.back().first + merged.back().second == r.first)
        merged.back().second += r.second;
      else
        merged.push_back(r);
    }
    fs->free_ranges.swap(merged);
  }

  // The graph of steps_per_launch steps with the smallest power-of-two grid (64 to kMaxFlowGrid) of at
  // least the resident runs: workgroups without a run would still be dispatched.  Each is captured
  // once, when first needed, which adds 0.25-0.45 ms to that call of dfrg_fs_progress (0.65 ms at 200 steps
  // per launch), at most five times in a server's life; creating them all beforehand would cost every
  // server as much as one that needs them all.
  int fs_capture(dfrg_fs *fs, hipGraphExec_t *exec)
  {
    const int R = *fs->mirror<int>(fs->sl.n_runs);
    int g = 0;
    while ((64 << g) < R && (64 << g) < kMaxFlowGrid) ++g;
    *exec = fs->graph_exec[g];
    if (*exec) return DFRG_OK;
    hipStream_t cs;
    DFRG_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    DFRG_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
    const size_t shm = sizeof(double2) * ((fs->nx + 63) / 64 * 64);
    for (int st = 0; st < fs->steps_per_launch; ++st)
      hipLaunchKernelGGL(flow_step_kernel, dim3(64 << g), dim3(kRunBlock), shm, cs, fs->dev, st);
    hipLaunchKernelGGL(flow_base_kernel, dim3(1), dim3(64), 0, cs, fs->dev.base, fs->steps_per_launch);
    hipGraph_t gr = nullptr;
    hipError_t e = hipStreamEndCapture(cs, &gr);
    hipStreamDestroy(cs);
    if (e != hipSuccess) {
      set_error("flow graph capture failed: %s", hipGetErrorString(e));
      return DFRG_ERR_HIP;
    }
    e = hipGraphInstantiate(&fs->graph_exec[g], gr, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      (void)hipGraphDestroy(gr);
      fs->graph_exec[g] = nullptr;
      set_error("flow graph instantiation failed: %s", hipGetErrorString(e));
      return DFRG_ERR_HIP;
    }
    fs->graph[g] = gr;
    *exec = fs->graph_exec[g];
    return DFRG_OK;
  }

  // retire finished / failed flows: copy u back, free their slot and HBM range
  int fs_retire(dfrg_fs *fs)
  {
    const int *bad = fs->mirror<int>(fs->sl.bad); // copied back behind the launch
    const double t = now_s();
    for (int s = 0; s < fs->max_resident; ++s) {
      if (fs->slot_flow[s] < 0) continue;
      FlowRecord &r = fs->flows[fs->slot_flow[s]];
      const bool done = fs->base - r.admit >= fs->n_steps;
      if (!done && !bad[s]) continue;
      const int n = r.desc.n_grid;
      r.u.resize(n);
      // u after the last step taken sits in the buffer of that step count's parity
      const int taken = std::min(fs->base - r.admit, fs->n_steps);
      const double *staged = nullptr;
      if (!bad[s])
        for (const auto &st : fs->u_staged)
          if (st.first == s) staged = fs->h_u + st.second;
      if (staged)
        std::copy(staged, staged + n, r.u.begin());
      else // a flow evicted as non-finite: its u after the last step taken
        DFRG_HIP(hipMemcpy(r.u.data(), fs->dev.pool + r.off + (taken & 1) * n, sizeof(double) * n,
                           hipMemcpyDeviceToHost));
      r.state = bad[s] ? 3 : 2;
      r.t_done = t;
      if (r.state == 2) {
        fs->latencies.push_back(r.t_done - r.t_submit);
        ++fs->finished;
      }
      fs_free_range(fs, r.off, 2 * n);
      fs->slot_flow[s] = -1;
      r.slot = -1;
      fs->runs_dirty = true;
    }
    return DFRG_OK;
  }

  int fs_admit(dfrg_fs *fs)
  {
    while (!fs->queue.empty()) {
      const long long id = fs->queue.front();
      FlowRecord &r = fs->flows[id];
      const int n = r.desc.n_grid;
      int slot = -1;
      for (int s = 0; s < fs->max_resident; ++s)
        if (fs->slot_flow[s] < 0) {
          slot = s;
          break;
        }
      if (slot < 0) break;
      const int off = fs_alloc_range(fs, 2 * n);
      if (off < 0) break; // does not fit the HBM budget now: wait for retirements (FIFO)
      fs->queue.pop_front();
      // step 0 reads the initial condition from the run records, and writes the odd buffer, so the
      // flow's HBM range needs no initialisation
      fs->mirror<int>(fs->sl.bad)[slot] = 0;
      fs->slots_dirty = true;
      fs->slot_flow[slot] = id;
      r.slot = slot;
      r.off = off;
      r.admit = fs->base;
      r.state = 1;
      fs->runs_dirty = true;
    }
    if (fs->runs_dirty) {
      // cut every resident flow into runs of at most L points (and at least 2).  A workgroup holds 64
      // points of a stage at eight lanes per integral, 32 or 16 at 16 or 32, and a run's first stage
      // has L + 6; the L whose step is cheapest: per round of one workgroup on each CU a fixed part (its
      // first loads, about 250 instruction slots a stage) and the VALU instructions of a SIMD's waves
      // (155, 220 and 350 per stage for waves of one, two and four points)
      std::vector<int> sizes;
      for (int s = 0; s < fs->max_resident; ++s)
        if (fs->slot_flow[s] >= 0) sizes.push_back(fs->flows[fs->slot_flow[s]].desc.n_grid);
      const long long cus = context().cu_count > 0 ? context().cu_count : 256;
      auto pieces = [](int n, int len) { return std::min((n + len - 1) / len, n / 2); };
      int L = kMaxRun;
      double best = 1e300;
      for (int len : kRunLengths) {
        long long c = 0;
        for (int n : sizes) c += pieces(n, len);
        const int first = len + 2 * kHalo;
        const int issue = first <= 16   ? (first + 3) / 4 * 155
                          : first <= 32 ? (first + 7) / 8 * 220
                                        : (first + 15) / 16 * 350;
        const double cost = (double)((c + cus - 1) / cus) * (250 + issue);
        if (cost < best) {
          best = cost;
          L = len;
        }
      }
      std::vector<FlowRun> runs;
      for (int s = 0; s < fs->max_resident; ++s) {
        if (fs->slot_flow[s] < 0) continue;
        const FlowRecord &r = fs->flows[fs->slot_flow[s]];
        const int n = r.desc.n_grid, cnt = pieces(n, L), len = n / cnt, extra = n % cnt;
        const double h = r.desc.rho_max / (n - 1);
        for (int j = 0, a = 0; j < cnt; ++j) {
          const int b = a + len + (j < extra ? 1 : 0);
          runs.push_back(FlowRun{s, a, b, n, r.off, r.admit, h, 0.5 / h, 1.0 / (h * h), r.desc.T, r.desc.N,
                                 r.desc.m2_0, r.desc.lambda});
          a = b;
        }
      }
      const int R = (int)runs.size();
      if ((size_t)R > fs->runs_cap) {
        set_error("internal: %d flow runs exceed the %zu allocated", R, fs->runs_cap);
        return DFRG_ERR_RUNTIME;
      }
      // staged in pinned memory and uploaded before the next launch (no copy is in flight here:
      // every launch ends with a synchronisation)
      if ((size_t)R > fs->h_runs_cap) {
        const size_t cap = std::max<size_t>((size_t)R, 2 * fs->h_runs_cap);
        if (fs->h_runs) (void)hipHostFree(fs->h_runs);
        fs->h_runs = nullptr;
        fs->h_runs_cap = 0;
        DFRG_HIP(hipHostMalloc((void **)&fs->h_runs, sizeof(FlowRun) * cap, hipHostMallocDefault));
        fs->h_runs_cap = cap;
      }
      if (R) std::copy(runs.begin(), runs.end(), fs->h_runs);
      fs->runs_upload = R;
      *fs->mirror<int>(fs->sl.n_runs) = R;
      fs->slots_dirty = true;
      fs->runs_dirty = false;
    }
    return DFRG_OK;
  }

  int resident_count(const dfrg_fs *fs)
  {
    int c = 0;
    for (long long id : fs->slot_flow) c += id >= 0;
    return c;
  }
} // namespace

extern "C" {

size_t dfrg_fs_flow_bytes(int n_grid) { return (size_t)2 * n_grid * sizeof(double); }

int dfrg_fs_timing(dfrg_fs *fs, long long *launches, double *device_s, long long *point_steps)
{
  DFRG_CHECK_ARG(fs != nullptr, "NULL server");
  if (launches) *launches = fs->launches;
  if (device_s) *device_s = fs->device_s;
  if (point_steps) *point_steps = fs->point_steps;
  return DFRG_OK;
}

int dfrg_fs_create(dfrg_fs **out, dfrg_qp *qp, size_t hbm_budget, int max_resident, int nx, int n_steps,
                   double k_end, int steps_per_launch)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(out && qp, "NULL handle");
  DFRG_CHECK_ARG(max_resident >= 1 && max_resident <= 4096, "max_resident %d out of range [1,4096]", max_resident);
  DFRG_CHECK_ARG(nx >= 1 && nx <= 1024, "nx %d out of range", nx);
  DFRG_CHECK_ARG(n_steps >= 1 && k_end > 0 && k_end < 1, "invalid n_steps / k_end");
  DFRG_CHECK_ARG(steps_per_launch >= 1 && steps_per_launch <= 1000, "steps_per_launch out of range");
  const size_t max_points = (size_t)max_resident * 4096;
  DFRG_CHECK_ARG(hbm_budget >= dfrg_fs_flow_bytes(4) && hbm_budget / sizeof(double) < (size_t)1 << 31,
                 "hbm_budget out of range");
  dfrg_fs *fs = new dfrg_fs;
  fs->budget = hbm_budget;
  fs->max_resident = max_resident;
  fs->nx = nx;
  fs->n_steps = n_steps;
  fs->k_end = k_end;
  fs->steps_per_launch = steps_per_launch;
  fs->pool_doubles = hbm_budget / sizeof(double);
  fs->free_ranges.push_back({0, (int)fs->pool_doubles});
  fs->slot_flow.assign(max_resident, -1);
  FlowDev &d = fs->dev;
  d.nx = nx;
  d.n_steps = n_steps;
  d.dt = std::log(1.0 / k_end) / n_steps;
  const void *hx = nullptr, *hw = nullptr;
  int rc = dfrg_qp_gl(qp, nx, 0, nullptr, nullptr, &hx, &hw);
  if (rc != DFRG_OK) {
    delete fs;
    return rc;
  }
  // node factors and k(t) (header comment); k as the oracle's stepper forms it: t = s dt,
  // exp(-t), exp(-(t + dt/2)), exp(-(t + dt))
  const int nxp = (nx + 63) / 64 * 64;
  std::vector<double> nodes(2 * nxp + kFlowExp + 3 * (size_t)n_steps);
  for (int j = 0; j < nx; ++j) {
    const double xr = ((const double *)hx)[j] * fs->x_extent;
    const double e = std::exp(-xr);
    nodes[2 * j] = xr + e;
    nodes[2 * j + 1] =
        0.25 * (std::sqrt(xr) * (((const double *)hw)[j] * fs->x_extent) * e * (1.0 + xr) / (2.0 * kPi * kPi));
  }
  for (int j = nx; j < nxp; ++j) nodes[2 * j] = 1e30;
  // 2^(j/512) as products of 32 and 16 extended-precision values (the same 512 doubles as one exp2l
  // each, which takes the host 30-57 us against 4)
  long double coarse[kFlowExp / 16], fine[16];
  for (int j = 0; j < kFlowExp / 16; ++j) coarse[j] = std::exp2((long double)j * 16 / kFlowExp);
  for (int j = 0; j < 16; ++j) fine[j] = std::exp2((long double)j / kFlowExp);
  for (int j = 0; j < kFlowExp; ++j) nodes[2 * nxp + j] = (double)(coarse[j / 16] * fine[j % 16]);
  double *kt = &nodes[2 * nxp + kFlowExp];
  for (int st = 0; st < n_steps; ++st) {
    const double t = st * d.dt;
    kt[3 * st] = std::exp(-t);
    kt[3 * st + 1] = std::exp(-(t + 0.5 * d.dt));
    kt[3 * st + 2] = std::exp(-(t + d.dt));
  }
  // runs: at least 2 points each, and a resident flow of n points holds 2 n doubles of the pool
  fs->runs_cap = std::max<size_t>(std::min(max_points, fs->pool_doubles / 4 + (size_t)max_resident + 1), kMaxFlowGrid);
  const size_t runs_bytes = sizeof(FlowRun) * fs->runs_cap;
#define FS_ALLOC(ptr, bytes)                                                                                   \
  do {                                                                                                         \
    if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess || hipMemset((ptr), 0, (bytes)) != hipSuccess) {     \
      set_error("flow server: device allocation of %zu bytes failed", (size_t)(bytes));                        \
      dfrg_fs_destroy(fs);                                                                                     \
      return DFRG_ERR_HIP;                                                                                     \
    }                                                                                                          \
  } while (0)
  {
    SlotLayout &L = fs->sl;
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t M = (size_t)max_resident;
    size_t o = 0;
    L.n_runs = o, o += up(sizeof(int));
    L.bad = o, o += up(sizeof(int) * M);
    L.bytes = o;
  }
  FS_ALLOC(fs->d_slots, fs->sl.bytes);
  if (hipHostMalloc((void **)&fs->h_slots, fs->sl.bytes, hipHostMallocDefault) != hipSuccess) {
    fs->h_slots = nullptr;
    set_error("flow server: pinned allocation of %zu bytes failed", fs->sl.bytes);
    dfrg_fs_destroy(fs);
    return DFRG_ERR_HIP;
  }
  std::memset(fs->h_slots, 0, fs->sl.bytes);
  d.n_runs = (int *)(fs->d_slots + fs->sl.n_runs);
  d.bad = (int *)(fs->d_slots + fs->sl.bad);
  FS_ALLOC(d.runs, runs_bytes);
  FS_ALLOC(d.base, sizeof(int));
  FS_ALLOC(fs->d_nodes, sizeof(double) * nodes.size());
  FS_ALLOC(d.pool, sizeof(double) * fs->pool_doubles);
#undef FS_ALLOC
  d.nodes = (const double2 *)fs->d_nodes;
  d.exp2t = fs->d_nodes + 2 * nxp;
  d.kt = fs->d_nodes + 2 * nxp + kFlowExp;
  if (hipMemcpy(fs->d_nodes, nodes.data(), sizeof(double) * nodes.size(), hipMemcpyHostToDevice) != hipSuccess) {
    set_error("flow server: node table upload failed");
    dfrg_fs_destroy(fs);
    return DFRG_ERR_HIP;
  }
  if (hipStreamCreateWithFlags(&fs->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&fs->ev0) != hipSuccess || hipEventCreate(&fs->ev1) != hipSuccess) {
    set_error("flow server: stream creation failed");
    dfrg_fs_destroy(fs);
    return DFRG_ERR_HIP;
  }
  DFRG_HIP(hipDeviceSynchronize());
  *out = fs;
  return DFRG_OK;
}

int dfrg_fs_destroy(dfrg_fs *fs)
{
  if (!fs) return DFRG_OK;
  hipDeviceSynchronize();
  for (int g = 0; g < kFlowGraphs; ++g) {
    if (fs->graph_exec[g]) hipGraphExecDestroy(fs->graph_exec[g]);
    if (fs->graph[g]) hipGraphDestroy(fs->graph[g]);
  }
  if (fs->ev0) hipEventDestroy(fs->ev0);
  if (fs->ev1) hipEventDestroy(fs->ev1);
  if (fs->stream) hipStreamDestroy(fs->stream);
  FlowDev &d = fs->dev;
  for (void *p : {(void *)fs->d_slots, (void *)d.runs, (void *)d.base, (void *)d.pool, (void *)fs->d_nodes})
    if (p) hipFree(p);
  for (void *p : {(void *)fs->h_slots, (void *)fs->h_runs, (void *)fs->h_u})
    if (p) hipHostFree(p);
  delete fs;
  return DFRG_OK;
}

int dfrg_fs_submit(dfrg_fs *fs, const dfrg_flow_desc *desc, long long *id)
{
  DFRG_CHECK_ARG(fs && desc && id, "NULL argument");
  DFRG_CHECK_ARG(desc->n_grid >= 4 && desc->n_grid <= 4096, "n_grid %d out of range [4,4096]", desc->n_grid);
  DFRG_CHECK_ARG(desc->rho_max > 0 && desc->T > 0 && desc->N >= 1, "invalid flow parameters");
  DFRG_CHECK_ARG(std::isfinite(desc->m2_0) && std::isfinite(desc->lambda) && std::isfinite(desc->mu),
                 "invalid flow parameters");
  DFRG_CHECK_ARG(dfrg_fs_flow_bytes(desc->n_grid) <= fs->budget, "flow of %d points exceeds the HBM budget",
                 desc->n_grid);
  FlowRecord r;
  r.desc = *desc;
  r.t_submit = now_s();
  const long long fid = fs->next_id++;
  fs->flows.emplace(fid, std::move(r));
  fs->queue.push_back(fid);
  *id = fid;
  return DFRG_OK;
}

int dfrg_fs_progress(dfrg_fs *fs, int *resident, int *queued, int *done)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(fs != nullptr, "NULL server");
  DFRG_TRY(fs_admit(fs));
  if (resident_count(fs) > 0) {
    hipGraphExec_t graph = nullptr;
    DFRG_TRY(fs_capture(fs, &graph));
    // grid-point steps this launch advances: each resident flow takes the steps it has left, up to
    // steps_per_launch
    for (long long id : fs->slot_flow)
      if (id >= 0) {
        const FlowRecord &r = fs->flows[id];
        const int left = fs->n_steps - (fs->base - r.admit);
        fs->point_steps += (long long)r.desc.n_grid * std::max(0, std::min(left, fs->steps_per_launch));
      }
    // pinned staging for the final u of the flows that take their last step in this launch (no
    // copy is in flight here: the previous launch ended with a synchronisation)
    size_t need = 0;
    for (long long id : fs->slot_flow)
      if (id >= 0) {
        const FlowRecord &r = fs->flows[id];
        if (fs->base + fs->steps_per_launch - r.admit >= fs->n_steps) need += r.desc.n_grid;
      }
    if (need > fs->h_u_cap) {
      const size_t cap = std::max(need, 2 * fs->h_u_cap);
      if (fs->h_u) (void)hipHostFree(fs->h_u);
      fs->h_u = nullptr;
      fs->h_u_cap = 0;
      DFRG_HIP(hipHostMalloc((void **)&fs->h_u, sizeof(double) * cap, hipHostMallocDefault));
      fs->h_u_cap = cap;
    }
    const double t0 = now_s();
    // the slot block and run table go up asynchronously from their pinned staging
    if (fs->slots_dirty) {
      DFRG_HIP(hipMemcpyAsync(fs->d_slots, fs->h_slots, fs->sl.bytes, hipMemcpyHostToDevice, fs->stream));
      fs->slots_dirty = false;
    }
    if (fs->runs_upload > 0)
      DFRG_HIP(hipMemcpyAsync(fs->dev.runs, fs->h_runs, sizeof(FlowRun) * fs->runs_upload, hipMemcpyHostToDevice,
                              fs->stream));
    fs->runs_upload = 0;
    DFRG_HIP(hipEventRecord(fs->ev0, fs->stream));
    DFRG_HIP(hipGraphLaunch(graph, fs->stream));
    DFRG_HIP(hipEventRecord(fs->ev1, fs->stream));
    // behind the graph: the non-finite flags into the mirror, and the finishers' final u
    DFRG_HIP(hipMemcpyAsync(fs->h_slots + fs->sl.bad, fs->dev.bad, sizeof(int) * fs->max_resident,
                            hipMemcpyDeviceToHost, fs->stream));
    fs->u_staged.clear();
    size_t o = 0;
    for (int sl = 0; sl < fs->max_resident; ++sl) {
      const long long id = fs->slot_flow[sl];
      if (id < 0) continue;
      const FlowRecord &r = fs->flows[id];
      if (fs->base + fs->steps_per_launch - r.admit < fs->n_steps) continue;
      const int n = r.desc.n_grid; // u after the last step sits in the buffer of n_steps' parity
      DFRG_HIP(hipMemcpyAsync(fs->h_u + o, fs->dev.pool + r.off + (fs->n_steps & 1) * n, sizeof(double) * n,
                              hipMemcpyDeviceToHost, fs->stream));
      fs->u_staged.push_back({sl, o});
      o += n;
    }
    DFRG_HIP(hipStreamSynchronize(fs->stream));
    fs->base += fs->steps_per_launch;
    fs->busy_s += now_s() - t0;
    float ms = 0.f;
    DFRG_HIP(hipEventElapsedTime(&ms, fs->ev0, fs->ev1));
    fs->device_s += 1e-3 * ms;
    ++fs->launches;
    DFRG_TRY(fs_retire(fs));
    DFRG_TRY(fs_admit(fs));
  }
  if (resident) *resident = resident_count(fs);
  if (queued) *queued = (int)fs->queue.size();
  if (done) *done = fs->finished;
  return DFRG_OK;
}

int dfrg_fs_poll(dfrg_fs *fs, long long id, int *state)
{
  DFRG_CHECK_ARG(fs && state, "NULL argument");
  auto it = fs->flows.find(id);
  DFRG_CHECK_ARG(it != fs->flows.end(), "unknown flow id %lld", id);
  *state = it->second.state;
  return DFRG_OK;
}

int dfrg_fs_result(dfrg_fs *fs, long long id, double *u_out, int n, double *latency_s)
{
  DFRG_CHECK_ARG(fs && u_out, "NULL argument");
  auto it = fs->flows.find(id);
  DFRG_CHECK_ARG(it != fs->flows.end(), "unknown flow id %lld", id);
  FlowRecord &r = it->second;
  DFRG_CHECK_ARG(r.state == 2 || r.state == 3, "flow %lld has not finished", id);
  DFRG_CHECK_ARG(n >= r.desc.n_grid, "output holds %d < %d points", n, r.desc.n_grid);
  std::copy(r.u.begin(), r.u.end(), u_out);
  if (latency_s) *latency_s = r.t_done - r.t_submit;
  const int failed = r.state == 3;
  fs->flows.erase(it);
  if (failed) {
    set_error("flow %lld became non-finite", id);
    return DFRG_ERR_RUNTIME;
  }
  return DFRG_OK;
}

int dfrg_fs_stats(dfrg_fs *fs, int *finished, double *p50_s, double *p99_s, double *busy_s)
{
  DFRG_CHECK_ARG(fs != nullptr, "NULL server");
  std::vector<double> l = fs->latencies;
  std::sort(l.begin(), l.end());
  auto pct = [&](double p) {
    if (l.empty()) return 0.0;
    const double pos = p * (l.size() - 1);
    const size_t i0 = (size_t)pos;
    const size_t i1 = std::min(i0 + 1, l.size() - 1);
    return l[i0] + (pos - i0) * (l[i1] - l[i0]);
  };
  if (finished) *finished = fs->finished;
  if (p50_s) *p50_s = pct(0.50);
  if (p99_s) *p99_s = pct(0.99);
  if (busy_s) *busy_s = fs->busy_s;
  return DFRG_OK;
}

} // extern "C"
