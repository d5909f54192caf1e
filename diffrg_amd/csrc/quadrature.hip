// quadrature.hip -- FP64 quadrature rules generated on the GPU, and the provider cache.
//
// Gauss-Legendre: one lane per root.  FP64 Newton iterations on the Legendre three-term recurrence
// bring the root to a few roundings; one compensated pass of the same recurrence (its rounding
// errors carried exactly and propagated alongside) then gives P_n there to twice FP64's digits, so
// that nodes near 0 and 1 keep full relative precision after the map t = (1 -+ z)/2.  Replaces GSL's
// gsl_integration_fixed_legendre (quadrature.cu:23-58).
//
// Matsubara (Monien, Math. Comp. 79, 857 (2010); matsubara.cu:33-85): the Jacobi matrix of the
// recurrence a_j, b_j; wave i finds the i-th smallest eigenvalue by multisection on the Sturm count
// (64 points per round) and the first component of its eigenvector from a twisted factorisation
// (Parlett & Dhillon's twisted LDL^T / UDU^T, the core of MRRR).  The reference diagonalises the
// same matrix with the sequential implicit-QL routine IMTQLX (diagonalization.hh:34-145); the
// parallel form is at least as accurate on this graded matrix.
#include "internal.hh"
#include "dfrg/device.hh"

// The compensated recurrence below relies on error-free transformations; fusing a product
// into a later sum (FP contraction, on by default for device code) would break them.
#pragma clang fp contract(off)

#include <cmath>
#include <map>
#include <vector>

namespace dfrg
{
  namespace
  {
    // a + b = sum + err exactly (Knuth)
    __device__ __forceinline__ double two_sum(double a, double b, double &err)
    {
      const double s = a + b;
      const double bb = s - a;
      err = (a - (s - bb)) + (b - bb);
      return s;
    }

    // Rules of a few dozen to a few hundred nodes run on a handful of waves, so the serial recurrence
    // over the order bounds the kernel: what counts is its dependent chain per degree.  With 1/j
    // tabulated in LDS, an FP64 step is one dependent FMA, and the compensated step has four
    // dependent operations with its error terms beside them; the earlier form took every Newton step
    // in double-double with a three-division quotient per degree.  Order 128: 293 -> 16.8 us, 32: 86 ->
    // 6.6, 1024: 1972 -> 96.5.  LONG, for orders past kGlTable (half a long vacuum rule): the reciprocals of the
    // further degrees are formed in the step (one kernel for both: 2% slower up to kGlTable).
    constexpr int kGlBlock = 64;
    constexpr int kGlTable = 4096; // 64 KB of LDS
    // 1/j = x + y
    __device__ __forceinline__ double2 gl_inverse(int j)
    {
      const double hi = 1.0 / j;
      return make_double2(hi, fma(-hi, (double)j, 1.0) * hi);
    }
    template <bool LONG> __global__ __launch_bounds__(kGlBlock) void gl_kernel(int n, double *x, double *w)
    {
      extern __shared__ double2 s_inv[]; // 1/j at j - 1, j <= n_tab
      const int n_tab = LONG ? kGlTable : n;
      for (int j = 1 + threadIdx.x; j <= n_tab; j += kGlBlock) s_inv[j - 1] = gl_inverse(j);
      __syncthreads();
      const int i = blockIdx.x * kGlBlock + threadIdx.x;
      const bool own = i < (n + 1) / 2;
      // i-th root from the top; Tricomi's initial guess.  Odd n: the middle root is 0 exactly.
      const double dn = n;
      const bool middle = (n & 1) && i == n / 2;
      double z = middle || !own ? 0.0
                                : (1.0 - (dn - 1.0) / (8.0 * dn * dn * dn)) * cos(dev::pi * (i + 0.75) / (n + 0.5));
      // Newton in FP64: P_j = (2 - 1/j) z P_{j-1} - (1 - 1/j) P_{j-2};  P_n' = n (z P_n - P_{n-1})/(z^2 - 1)
      for (int it = 0; it < 8; ++it) {
        double p0 = 1.0, p1 = z;
        auto step = [&](double inv) {
          const double p2 = fma((2.0 - inv) * z, p1, -((1.0 - inv) * p0));
          p0 = p1;
          p1 = p2;
        };
#pragma unroll 8
        for (int j = 2; j <= n_tab; ++j) step(s_inv[j - 1].x);
        if (LONG)
          for (int j = kGlTable + 1; j <= n; ++j) step(gl_inverse(j).x);
        const double dz = p1 * fma(z, z, -1.0) / (dn * fma(z, p1, -p0));
        if (n > 1 && own && !middle) z -= dz;
        // the step leaves about dz^2 n^2/6 near the ends, less elsewhere: below an FP64 rounding
        if (__builtin_amdgcn_ballot_w64(own && !middle && fabs(dz) * dn > 3e-8) == 0) break;
      }
      // one pass at the FP64 root with its rounding errors: with u = z P_{j-1} and t = u - P_{j-2},
      // P_j = u + t - t/j; e carries the error of P_j through the same recurrence
      double p0 = 1.0, p1 = z, e0 = 0.0, e1 = 0.0;
      auto step = [&](double2 inv) {
        double dt, ds, dp;
        const double u = z * p1, du = fma(z, p1, -u);
        const double t = two_sum(u, -p0, dt);
        const double v = t * inv.x, dv = fma(t, inv.x, -v);
        const double s = two_sum(u, t, ds);
        const double p2 = two_sum(s, -v, dp);
        const double eu = fma(z, e1, du), et = (eu - e0) + dt;
        const double ev = fma(et, inv.x, fma(t, inv.y, dv));
        const double e2 = ((eu + et) - ev) + (ds + dp);
        p0 = p1;
        p1 = p2;
        e0 = e1;
        e1 = e2;
      };
#pragma unroll 4
      for (int j = 2; j <= n_tab; ++j) step(s_inv[j - 1]);
      if (LONG)
        for (int j = kGlTable + 1; j <= n; ++j) step(gl_inverse(j));
      if (!own) return;
      const double f = n > 1 ? p1 + e1 : 0.0;
      if (n == 1) {
        p0 = 1.0;
        e0 = 0.0;
      }
      // 1 - z and 1 + z exactly, and the root's correction d: Newton with its second-order term
      // (P'' = 2 z P'/(1 - z^2) at a root)
      double om_e, op_e;
      const double om = two_sum(1.0, -z, om_e), op = two_sum(1.0, z, op_e);
      const double q = om * op;                                // 1 - z^2
      const double pm = p0 + e0;
      const double d1 = -f * q / (dn * fma(-z, f, pm)); // -P/P'
      const double d = middle ? 0.0 : d1 - d1 * d1 * (z / q);
      const double om_l = om_e - d, op_l = op_e + d;
      const double xlo = om + om_l, xhi = op + op_l; // 1 - z*, 1 + z*
      // weight on [0,1]: 1 / ((1 - z^2) P_n'(z)^2) = (1 - z^2) / (n P_{n-1})^2 at the root z* = z + d, in
      // twice FP64's digits up to the last division: P_{n-1} moved by its Taylor series (P'/P =
      // n (z - P_n/P)/(1 - z^2) =: g, P''/P = (2 z g - n (n - 1))/(1 - z^2))
      const double g = dn * (z - f / pm) / q, h = 0.5 * (2.0 * z * g - dn * (dn - 1.0)) / q;
      const double pm_l = fma(pm, fma(h, d, g) * d, e0);
      const double t = dn * p0, t_l = fma(dn, pm_l, fma(dn, p0, -t));
      const double den = t * t, den_l = fma(t, t, -den) + (2.0 * t * t_l + t_l * t_l);
      const double num = q, num_l = fma(om, op, -q) + (om * op_l + om_l * op);
      const double w0 = num / den;
      const double wz = w0 + (fma(-w0, den, num) + fma(-w0, den_l, num_l)) / (den + den_l);
      x[n - 1 - i] = 0.5 * xhi;
      x[i] = middle ? 0.5 : 0.5 * xlo;
      w[n - 1 - i] = wz;
      w[i] = wz;
    }

    // ---------------------------------------------------------------------------------------
    // Monien rule
    // ---------------------------------------------------------------------------------------
    // Number of eigenvalues of the tridiagonal (a, e^2) below x: negative pivots of its LDL^T
    // factorisation.
    __device__ __forceinline__ int sturm_count_below(const double2 *m, int n, double x)
    {
      double q = m[0].x - x;
      int c = q < 0.0;
#pragma unroll 4
      for (int j = 1; j < n; ++j) {
        if (q == 0.0) q = 1e-300;
        q = (m[j].x - x) - m[j].y / q;
        c += q < 0.0;
      }
      return c;
    }

    // The same count by the sign changes of the Sturm sequence p_j = (a_j - x) p_{j-1} - e_{j-1}^2 p_{j-2},
    // whose ratios are those pivots: one dependent FMA per step instead of a division, and the two agree
    // but for x within about 1e-12 of an eigenvalue.  The pair is rescaled by a power of two every
    // eight steps; the entries (e^2 down to 1e-13 at n = 1024) cannot take it out of range in between.
    __device__ __forceinline__ int sturm_count_quick(const double2 *m, int n, double x)
    {
      double p0 = 1.0, p1 = m[0].x - x;
      int c = p1 < 0.0;
      auto step = [&](int j) {
        const double2 ae = m[j]; // a_j, e_{j-1}^2
        double p2 = fma(ae.x - x, p1, -(ae.y * p0));
        if (p2 == 0.0) p2 = copysign(1e-200, p1); // a zero pivot counts as positive, the next as negative
        c += (unsigned)(__double2hiint(p2) ^ __double2hiint(p1)) >> 31;
        p0 = p1;
        p1 = p2;
      };
      int j = 1;
      for (; j + 8 <= n; j += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) step(j + u);
        const int ex = -max(__builtin_amdgcn_frexp_exp(p0), __builtin_amdgcn_frexp_exp(p1));
        p0 = ldexp(p0, ex);
        p1 = ldexp(p1, ex);
      }
      for (; j < n; ++j) step(j);
      return c;
    }

    // One wave per node: every block forms the matrix in its LDS.  Rounds of 64 points shrink the bracket
    // about 64-fold each, nine quick counts and two with pivots against 70 bisection steps with pivots,
    // whose division chain bounded the kernel (all nodes had shared one block); the two halves of the
    // twisted factorisation run on two lanes.  A provider's rule
    // of 66 nodes, call to result, 414 -> 50 us, of 32 nodes 213 -> 39.
    __global__ __launch_bounds__(64) void matsubara_kernel(int n, double T, double *x_out, double *w_out)
    {
      extern __shared__ double sm[];
      double2 *m = (double2 *)sm; // a_j, e_{j-1}^2
      double *e = sm + 2 * n;     // off-diagonal, e[j] couples j and j+1
      double *d = sm + 3 * n, *dp = sm + 4 * n;
      const double pi = dev::pi;
      const int lane = threadIdx.x, k = blockIdx.x;
      for (int j = lane; j < n; j += 64) {
        const double j1 = j + 1;
        double aj = 2.0 * (pi * pi) / (4 * j + 1) / (4 * j + 5);
        if (j == 0) aj = (pi * pi) / 15.0;
        const double bj = (pi * (pi * (pi * pi))) / ((4 * j1 - 1) * (4 * j1 + 3)) / ((4 * j1 + 1) * (4 * j1 + 1));
        const double ej = (j < n - 1) ? sqrt(bj) : 0.0;
        e[j] = ej;
        m[j].x = aj;
        if (j + 1 < n) m[j + 1].y = ej * ej;
        if (j == 0) m[0].y = 0.0;
      }
      __syncthreads();
      // k-th smallest eigenvalue, 64 points per round: count(x) > k  <=>  lambda_k < x.  All lie in (0, 2)
      // (Gershgorin); the first round's points are geometric, as the eigenvalues fall like 1/i^2 down to
      // n^-4.
      double lo = 0.0, hi = 2.0;
      auto narrow = [&](double x, int count) {
        const unsigned long long above = __builtin_amdgcn_ballot_w64(count > k);
        const int f = above ? __builtin_ctzll(above) : 64; // first point above the eigenvalue
        if (f < 64) hi = dev::lane_value(x, f);
        if (f > 0) lo = dev::lane_value(x, f - 1);
        return f;
      };
      {
        const double x = exp2(-40.0 + (lane + 1) * (41.0 / 65.0));
        narrow(x, sturm_count_quick(m, n, x));
      }
      for (int it = 0; it < 16 && hi - lo > 0x1p-40 * hi; ++it) {
        const double x = fma(hi - lo, (lane + 1) * (1.0 / 65.0), lo);
        narrow(x, sturm_count_quick(m, n, x));
      }
      // the last digits by the pivots, as the reference's accuracy is theirs: from a bracket of 1e-12 about
      // the quick count's value, moved outwards while the pivots' eigenvalue is not in it
      double w = 0x1p-41 * hi;
      lo -= w;
      hi += w;
      for (int it = 0; it < 16; ++it) {
        const double mid = 0.5 * (lo + hi);
        if (mid <= lo || mid >= hi || hi - lo <= 0x1p-51 * hi) break;
        const double x = fma(hi - lo, lane * (1.0 / 63.0), lo); // both ends among the points
        const double l0 = lo, h0 = hi;
        const int f = narrow(x, sturm_count_below(m, n, x));
        w *= 16.0;
        if (f == 0) lo = l0 - w;  // hi became the old lower end
        if (f == 64) hi = h0 + w; // lo became the old upper end
      }
      const double lam = 0.5 * (lo + hi);

      // twisted factorisation at lam: top-down pivots d on lane 0, bottom-up pivots dp on lane 1
      {
        double *out = lane == 0 ? d : dp;
        double q = m[lane == 0 ? 0 : n - 1].x - lam;
        if (lane < 2) out[lane == 0 ? 0 : n - 1] = q;
#pragma unroll 4
        for (int j = 1; j < n; ++j) {
          const int i = lane == 0 ? j : n - 1 - j;
          q = fma(-m[lane == 0 ? i : i + 1].y, dev::rcp_f64(q != 0.0 ? q : 1e-300), m[i].x - lam);
          if (lane < 2) out[i] = q;
        }
      }
      __syncthreads();
      // twist index: the smallest gamma_j, the first of equal ones
      int r = n;
      double gmin = INFINITY;
      for (int j = lane; j < n; j += 64) {
        const double g = fabs(d[j] + dp[j] - (m[j].x - lam));
        if (g < gmin) {
          gmin = g;
          r = j;
        }
      }
      for (int o = 32; o; o >>= 1) {
        const double g = __shfl_xor(gmin, o);
        const int ro = __shfl_xor(r, o);
        if (g < gmin || (g == gmin && ro < r)) {
          gmin = g;
          r = ro;
        }
      }
      r = __builtin_amdgcn_readfirstlane(r < n ? r : 0);
      // eigenvector with z_r = 1: ratios of neighbouring components (into d), then their products outward
      // from the twist index, downward indices on lane 0, upward ones on lane 1
      for (int j = lane; j < n; j += 64) {
        const double p = j < r ? d[j] : dp[j];
        d[j] = -((j < r ? e[j] : j > 0 ? e[j - 1] : 0.0) / (p != 0.0 ? p : 1e-300));
      }
      __syncthreads();
      double z = 1.0, s = 0.0;
      const int steps = lane == 0 ? r : n - 1 - r;
#pragma unroll 4
      for (int j = 1; j <= steps; ++j) {
        z *= d[lane == 0 ? r - j : r + j];
        s = fma(z, z, s);
      }
      const double z0 = dev::lane_value(z, 0);
      s = 1.0 + dev::lane_value(s, 0) + dev::lane_value(s, 1);
      if (lane != 0) return;
      const double mu0 = (pi * pi) / 6.0;
      const double wk = mu0 * (z0 * z0 / s);
      // normalise the weights and scale the nodes (matsubara.cu:78-84)
      w_out[k] = T * wk / lam;
      x_out[k] = 2.0 * pi * T / sqrt(lam);
    }

    // T = 0 rule (matsubara.cu:128-161): GL(h) on [0, 2E] and log-mapped GL(h) on [2E, 1e6 E].
    __global__ void matsubara_vacuum_kernel(int h, double E, const double *gx, const double *gw, double *x,
                                            double *w)
    {
      const int i = blockIdx.x * blockDim.x + threadIdx.x;
      if (i >= h) return;
      const double two_pi = 2.0 * dev::pi;
      const double div = 2.0 * fabs(E);
      x[i] = gx[i] * div;
      w[i] = gw[i] * div / two_pi;
      const double log_start = log(div);
      const double log_ext = log(1e6 * fabs(E) / div);
      const double xl = exp(log_start + log_ext * gx[i]);
      x[i + h] = xl;
      w[i + h] = (gw[i] * log_ext * xl) / two_pi;
    }

    // FP32 copies of a rule, and its host copies in pinned staging, behind the kernel that made it
    __global__ void rule_copies_kernel(int n, const double *x, const double *w, float *xf, float *wf, double *h)
    {
      const int i = blockIdx.x * blockDim.x + threadIdx.x;
      if (i >= n) return;
      const double xi = x[i], wi = w[i];
      xf[i] = (float)xi;
      wf[i] = (float)wi;
      h[i] = xi;
      h[n + i] = wi;
    }

    void launch_gl(int order, double *x, double *w, hipStream_t s)
    {
      const dim3 grid(((order + 1) / 2 + kGlBlock - 1) / kGlBlock);
      const size_t shm = sizeof(double2) * std::min(order, kGlTable);
      const auto kernel = order <= kGlTable ? gl_kernel<false> : gl_kernel<true>;
      hipLaunchKernelGGL(kernel, grid, dim3(kGlBlock), shm, s, order, x, w);
    }

    bool is_close_abs(double a, double b, double eps)
    {
      const double diff = std::fabs(a - b);
      return diff <= eps || diff <= std::fmax(std::fabs(a), std::fabs(b)) * eps;
    }

    // MatsubaraQuadrature::predict_size (matsubara.cu:12-21)
    int predict_size(double T, double E, int step, int vacuum_quad_size, int precision_factor)
    {
      const double rel = std::fabs(E) / std::fabs(T + 1e-16);
      if (is_close_abs(T, 0.0, 2.220446049250313e-16) || rel > 1e+2) return -vacuum_quad_size;
      const double E_max = (precision_factor + 100) * std::fabs(E);
      int size = 5 + (int)std::sqrt(4.0 * E_max / (M_PI * M_PI * std::fabs(T)));
      size = (int)std::ceil(size / (double)step) * step;
      return size;
    }
  } // namespace
} // namespace dfrg

using namespace dfrg;

namespace
{
  // dfrg_matsubara_generate without its synchronisation
  int enqueue_matsubara(double T, double E, int step, int min_size, int max_size, int vacuum_quad_size,
                        int precision_factor, double *d_x, double *d_w, int cap, int *size, double *T_rule,
                        hipStream_t s)
  {
    DFRG_CHECK_ARG(step >= 1, "step must be positive");
    DFRG_CHECK_ARG(std::isfinite(T) && std::isfinite(E) && T >= 0.0, "invalid T=%g / E=%g", T, E);
    if (precision_factor < 0) precision_factor = 1;
    if (vacuum_quad_size <= 6) vacuum_quad_size = 6;
    int m = predict_size(T, E, step, vacuum_quad_size, precision_factor);
    if (m < 0) {
      m = -m;
      if (m % 2) ++m;
      DFRG_CHECK_ARG(m <= cap, "vacuum Matsubara rule of %d nodes exceeds capacity %d", m, cap);
      if (is_close_abs(E, 0.0, 2.220446049250313e-16)) E = 1.0;
      const int h = m / 2;
      double *g = nullptr;
      DFRG_HIP(hipMallocAsync((void **)&g, sizeof(double) * 2 * h, s));
      launch_gl(h, g, g + h, s);
      DFRG_LAUNCHED("gl_kernel");
      hipLaunchKernelGGL(matsubara_vacuum_kernel, dim3(h / 64 + 1), dim3(64), 0, s, h, E, g, g + h, d_x, d_w);
      DFRG_LAUNCHED("matsubara_vacuum_kernel");
      DFRG_HIP(hipFreeAsync(g, s));
      *size = m;
      if (T_rule) *T_rule = 0.0;
      return DFRG_OK;
    }
    m = std::max(min_size, std::min(max_size, m));
    DFRG_CHECK_ARG(m >= 1 && m <= 1024, "Matsubara rule size %d out of range [1,1024]", m);
    DFRG_CHECK_ARG(m <= cap, "Matsubara rule of %d nodes exceeds capacity %d", m, cap);
    hipLaunchKernelGGL(matsubara_kernel, dim3(m), dim3(64), 5 * m * sizeof(double), s, m, T, d_x, d_w);
    DFRG_LAUNCHED("matsubara_kernel");
    *size = m;
    if (T_rule) *T_rule = T;
    return DFRG_OK;
  }
} // namespace

extern "C" {

int dfrg_gl_generate(int order, double *d_x, double *d_w, void *stream)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(order >= 1 && order <= 4096, "Gauss-Legendre order %d out of range [1,4096]", order);
  DFRG_CHECK_ARG(d_x && d_w, "output pointers are NULL");
  launch_gl(order, d_x, d_w, resolve_stream(stream));
  DFRG_LAUNCHED("gl_kernel");
  return DFRG_OK;
}

int dfrg_matsubara_generate(double T, double E, int step, int min_size, int max_size, int vacuum_quad_size,
                            int precision_factor, double *d_x, double *d_w, int cap, int *size, double *T_rule,
                            void *stream)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(d_x && d_w && size, "output pointers are NULL");
  hipStream_t s = resolve_stream(stream);
  DFRG_TRY(enqueue_matsubara(T, E, step, min_size, max_size, vacuum_quad_size, precision_factor, d_x, d_w, cap, size,
                             T_rule, s));
  DFRG_HIP(hipStreamSynchronize(s));
  return DFRG_OK;
}

} // extern "C"

// ---------------------------------------------------------------------------------------------
// provider cache (QuadratureProvider, quadrature_provider.hh:138-248, .cu:12-160)
// ---------------------------------------------------------------------------------------------
struct Rule {
  int size = 0;
  double T_rule = 0.0;
  double *d_x = nullptr, *d_w = nullptr;
  float *d_xf = nullptr, *d_wf = nullptr;
  std::vector<double> hx, hw;
  std::vector<float> hxf, hwf;
};

struct dfrg_qp {
  std::mutex mutex;
  // The rules' device memory: a few large blocks instead of four allocations per rule, given back when
  // the provider is destroyed.
  std::vector<char *> slabs;
  size_t slab_used = 0, slab_cap = 0;
  int vacuum_quad_size = 48;
  int min_matsubara_size = 32;
  int add_matsubara_size = 0;
  std::map<int, Rule> gl;
  std::map<double, std::map<double, Rule>> mats;
};

namespace
{
  // Room for a rule of up to cap nodes: x, w (FP64), then their FP32 copies.
  int place_rule(dfrg_qp *qp, Rule &r, int cap)
  {
    const size_t c = ((size_t)cap + 31) / 32 * 32, need = c * 2 * (sizeof(double) + sizeof(float));
    if (qp->slabs.empty() || qp->slab_used + need > qp->slab_cap) {
      const size_t bytes = std::max<size_t>(need, 64 << 10);
      void *p = nullptr;
      DFRG_HIP(hipMalloc(&p, bytes));
      qp->slabs.push_back((char *)p);
      qp->slab_used = 0;
      qp->slab_cap = bytes;
    }
    char *p = qp->slabs.back() + qp->slab_used;
    qp->slab_used += need;
    r.d_x = (double *)p;
    r.d_w = r.d_x + c;
    r.d_xf = (float *)(r.d_w + c);
    r.d_wf = r.d_xf + c;
    return DFRG_OK;
  }

  // Gives the room of the rule placed last back (a rule that could not be made); returns rc.  Kernels of the
  // rule may have been launched on s: the room is free when they have finished.
  int unplace_rule(dfrg_qp *qp, const Rule &r, int rc, hipStream_t s)
  {
    (void)hipStreamSynchronize(s);
    qp->slab_used = (size_t)((char *)r.d_x - qp->slabs.back());
    return rc;
  }

  // The copies of the rule in flight on s, and the wait for it: one kernel, one synchronisation.
  int finish_rule(Rule &r, hipStream_t s)
  {
    const int n = r.size;
    void *h = nullptr, *dh = nullptr;
    DFRG_TRY(dfrg_pool_host_alloc(&h, 2 * sizeof(double) * n));
    auto work = [&]() -> int {
      DFRG_HIP(hipHostGetDevicePointer(&dh, h, 0));
      hipLaunchKernelGGL(rule_copies_kernel, dim3((n + 63) / 64), dim3(64), 0, s, n, r.d_x, r.d_w, r.d_xf, r.d_wf,
                         (double *)dh);
      DFRG_LAUNCHED("rule_copies_kernel");
      return DFRG_OK;
    };
    int rc = work();
    // whatever was launched has finished before the staging goes back to its pool
    const hipError_t e = hipStreamSynchronize(s);
    if (rc == DFRG_OK && e != hipSuccess) {
      set_error("quadrature rule: %s", hipGetErrorString(e));
      rc = DFRG_ERR_HIP;
    }
    if (rc == DFRG_OK) {
      const double *v = (const double *)h;
      r.hx.assign(v, v + n);
      r.hw.assign(v + n, v + 2 * n);
      r.hxf.assign(r.hx.begin(), r.hx.end());
      r.hwf.assign(r.hw.begin(), r.hw.end());
    }
    dfrg_pool_host_free(h);
    return rc;
  }

  void hand_out(const Rule &r, int fp32, const void **d_x, const void **d_w, const void **h_x, const void **h_w)
  {
    if (d_x) *d_x = fp32 ? (const void *)r.d_xf : (const void *)r.d_x;
    if (d_w) *d_w = fp32 ? (const void *)r.d_wf : (const void *)r.d_w;
    if (h_x) *h_x = fp32 ? (const void *)r.hxf.data() : (const void *)r.hx.data();
    if (h_w) *h_w = fp32 ? (const void *)r.hwf.data() : (const void *)r.hw.data();
  }

  // find_T / find_E (quadrature_provider.cu:31-60): lower_bound, then the entry itself or its
  // predecessor when within 1e-6 * key.
  template <typename Map> typename Map::iterator find_close(Map &m, double key)
  {
    auto it = m.lower_bound(key);
    if (it != m.end() && is_close_abs(it->first, key, 1e-6 * key)) return it;
    if (it != m.begin()) {
      auto p = std::prev(it);
      if (is_close_abs(p->first, key, 1e-6 * key)) return p;
    }
    return m.end();
  }
} // namespace

extern "C" {

int dfrg_qp_create(dfrg_qp **qp, int vacuum_quad_size, int min_matsubara_size, int add_matsubara_size)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(qp != nullptr, "qp is NULL");
  DFRG_CHECK_ARG(vacuum_quad_size > 0, "MatsubaraStorage: Vacuum quadrature size must be positive.");
  DFRG_CHECK_ARG(add_matsubara_size >= 0, "MatsubaraStorage: add_matsubara_size must be positive.");
  DFRG_CHECK_ARG(min_matsubara_size > 0, "MatsubaraStorage: min_matsubara_size must be positive.");
  dfrg_qp *p = new dfrg_qp;
  p->vacuum_quad_size = vacuum_quad_size;
  p->min_matsubara_size = min_matsubara_size;
  p->add_matsubara_size = add_matsubara_size;
  *qp = p;
  return DFRG_OK;
}

int dfrg_qp_destroy(dfrg_qp *qp)
{
  if (!qp) return DFRG_OK;
  DFRG_TRY(require_init());
  hipDeviceSynchronize();
  for (char *p : qp->slabs) hipFree(p);
  delete qp;
  return DFRG_OK;
}

int dfrg_qp_gl(dfrg_qp *qp, int order, int fp32, const void **d_x, const void **d_w, const void **h_x,
               const void **h_w)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(qp != nullptr, "qp is NULL");
  DFRG_CHECK_ARG(order >= 1 && order <= 4096, "Gauss-Legendre order %d out of range [1,4096]", order);
  std::lock_guard<std::mutex> lock(qp->mutex);
  auto it = qp->gl.find(order);
  if (it == qp->gl.end()) {
    Rule r;
    r.size = order;
    DFRG_TRY(place_rule(qp, r, order));
    hipStream_t s = resolve_stream(nullptr);
    int rc = dfrg_gl_generate(order, r.d_x, r.d_w, s);
    if (rc == DFRG_OK) rc = finish_rule(r, s);
    if (rc != DFRG_OK) return unplace_rule(qp, r, rc, s);
    it = qp->gl.emplace(order, std::move(r)).first;
  }
  hand_out(it->second, fp32, d_x, d_w, h_x, h_w);
  return DFRG_OK;
}

int dfrg_qp_matsubara(dfrg_qp *qp, double T, double E, int fp32, int *size, double *T_rule, const void **d_x,
                      const void **d_w, const void **h_x, const void **h_w)
{
  DFRG_TRY(require_init());
  DFRG_CHECK_ARG(qp != nullptr, "qp is NULL");
  DFRG_CHECK_ARG(std::isfinite(T) && T >= 0.0, "invalid temperature %g", T);
  std::lock_guard<std::mutex> lock(qp->mutex);
  auto tit = find_close(qp->mats, T);
  if (tit == qp->mats.end()) tit = qp->mats.emplace(T, std::map<double, Rule>()).first;
  auto &emap = tit->second;
  auto eit = find_close(emap, E);
  if (eit == emap.end()) {
    Rule r;
    const int cap = std::max(qp->vacuum_quad_size + 2, 130);
    DFRG_TRY(place_rule(qp, r, cap));
    hipStream_t s = resolve_stream(nullptr);
    // MatsubaraStorage::find_E_d: reinit(T_key, E, 2, min_matsubara_size, 128, vacuum_quad_size,
    // add_matsubara_size) (quadrature_provider.cu:52)
    int rc = enqueue_matsubara(tit->first, E, 2, qp->min_matsubara_size, 128, qp->vacuum_quad_size,
                               qp->add_matsubara_size, r.d_x, r.d_w, cap, &r.size, &r.T_rule, s);
    if (rc == DFRG_OK) rc = finish_rule(r, s);
    if (rc != DFRG_OK) return unplace_rule(qp, r, rc, s);
    eit = emap.emplace(E, std::move(r)).first;
  }
  if (size) *size = eit->second.size;
  if (T_rule) *T_rule = eit->second.T_rule;
  hand_out(eit->second, fp32, d_x, d_w, h_x, h_w);
  return DFRG_OK;
}

} // extern "C"
