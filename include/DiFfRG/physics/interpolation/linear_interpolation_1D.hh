// DiFfRG/physics/interpolation/linear_interpolation_1D.hh -- tabulated dressing function
// evaluated inside kernels (reference linear_interpolation_1D.hh:22-113, .cu:15-98).
//
// The table lives in host memory and in HBM.  Copies are non-owning views (the copy the
// integrator passes by value into a kernel); update() on a view throws, as in the reference.
// operator() is the FP64-capable software lerp on the coordinate's index, clamped to [0, n-1];
// on the device it reads the HBM copy.  It replaces both LinearInterpolator1D and the FP32
// texture interpolator TexLinearInterpolator1D of the reference.
//
// FP64 logarithmic coordinates on the device: the reference's index idx = log1p(u) (N-1)/a,
// u = (x - c)/b, costs an FP64 division and log1p per call.  Here it comes from a table of sub-cells:
// K per cell (K the smallest power of two with |a|/(K(N-1)) <= 1/32), each with the smaller 1 + u_r of its
// ends.  An FP32 log2 of the mantissa of 1 + u plus its exponent locates the sub-cell m, and
//   K idx = m + o + K(N-1)/a log1p(delta),  delta = (u - u_r)/(1 + u_r) in [0, 0.0318],
// o = 0 when the sub-cell's start is the smaller end (a > 0), else 1; log1p as a polynomial of degree 7
// (Chebyshev interpolation on the sub-cell's range, remainder 7e-17).  An estimate one sub-cell off
// (within ~1e-5 of a boundary) gives the same sum.  The index agrees with the reference's to its own
// FP64 rounding (~1e-14 of a cell); the clamp to [0, N-1] and the reference's NaN rule (fmax(0, fmin(NaN,
// N-1)): a NaN index takes the last point) give the ends: u <= -1 takes the first point when u = -1 and
// a > 0 (index -inf), the last point otherwise (NaN, or +inf for a < 0); N = 1, bias 0 and NaN bias
// have a NaN or zero-width index: the last point.  On the device u below -1 or NaN counts as -1, where
// the sum is past the first end for a > 0 and past the last for a < 0 whatever the bias, and an o of 1e300
// moves it past the last end where u is not -1 itself.  The device code has no branch on the grid, so a
// user KERNEL's loop-invariant lookups (at q alone) stay hoistable.  Biases beyond +-700 (exp
// overflows) and grids of more than 2^21 sub-cells per unit of log2 are refused.
//
// VALU issue bounds a KERNEL made of lookups, exponentials and divisions: with sub-cells of 1/4, an
// atanh series to z^17 and the sub-cell corrected by selects, 64 requests of {64, 32, 32} nodes took
// 33.9 us in the kernel, now 29.7 (155 -> 127 VALU instructions per node).
#pragma once

#include <cmath>
#include <limits>
#include <memory>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "dfrg/check.hh"
#include "dfrg/math.hh"
#include <DiFfRG/discretization/grid/coordinates.hh>

namespace DiFfRG
{
  template <typename NT, typename Coordinates> class LinearInterpolator1D
  {
    static_assert(Coordinates::dim == 1, "LinearInterpolator1D requires 1D coordinates");

  public:
    LinearInterpolator1D(const std::vector<NT> &data, const Coordinates &coordinates)
        : LinearInterpolator1D(data.data(), coordinates)
    {
      if (data.size() != coordinates.size()) throw std::runtime_error("Data and coordinates must have the same size");
    }
    LinearInterpolator1D(const Coordinates &coordinates)
        : LinearInterpolator1D(std::vector<NT>(coordinates.size(), NT(0)), coordinates)
    {
    }
    LinearInterpolator1D(const NT *in_data, const Coordinates &coordinates)
        : size(coordinates.size()), coordinates(coordinates), owner(true)
    {
      dfrg::ensure_device();
      if constexpr (kLogFP64) make_cells(); // may refuse the grid: before the table's allocation
      m_data = std::shared_ptr<NT[]>(new NT[size]);
      for (unsigned i = 0; i < size; ++i) m_data[i] = NT(in_data[i]);
      void *p = nullptr;
      // at least two points in HBM: a one-point table's lerp reads its point twice
      dfrg::check(dfrg_malloc(&p, sizeof(NT) * (size < 2 ? 2 : size)), "LinearInterpolator1D");
      device_data = std::shared_ptr<void>(p, [](void *q) { dfrg_free(q); });
      device_data_ptr = (const NT *)p;
      update();
    }
    LinearInterpolator1D(const LinearInterpolator1D &other)
        : size(other.size), coordinates(other.coordinates), m_data(other.m_data), device_data(other.device_data),
          device_data_ptr(other.device_data_ptr), owner(false), cells(other.cells), lc(other.lc)
    {
    }

    template <typename NT2> void update(const NT2 *data)
    {
      if (!owner) throw std::runtime_error("Cannot update data of non-owner interpolator");
      for (unsigned i = 0; i < size; ++i) m_data[i] = NT(data[i]);
      update();
    }
    void update()
    {
      if (!owner) throw std::runtime_error("Cannot update data of non-owner interpolator");
      dfrg::check(dfrg_memcpy_h2d((void *)device_data_ptr, m_data.get(), sizeof(NT) * size, nullptr),
                 "LinearInterpolator1D::update");
      if (size == 1)
        dfrg::check(dfrg_memcpy_h2d((void *)(device_data_ptr + 1), m_data.get(), sizeof(NT), nullptr),
                    "LinearInterpolator1D::update");
      dfrg::check(dfrg_stream_sync(nullptr), "LinearInterpolator1D::update");
    }

    NT *data() const { return m_data.get(); }
    NT &operator[](const unsigned i) { return m_data[i]; }
    const NT &operator[](const unsigned i) const { return m_data[i]; }
    const Coordinates &get_coordinates() const { return coordinates; }

    __host__ __device__ NT operator()(const typename Coordinates::ctype x) const
    {
      using ct = typename Coordinates::ctype;
#ifdef __HIP_DEVICE_COMPILE__
      if constexpr (kLogFP64) return log_cell_lerp((x - lc.c) * lc.inv_b);
#endif
      ct idx = coordinates.backward(x);
      idx = fmax(ct(0), fmin(idx, ct(size - 1)));
      const ct fl = floor(idx);
#ifdef __HIP_DEVICE_COMPILE__
      const NT *d = device_data_ptr;
#else
      const NT *d = m_data.get();
#endif
      return dfrg::tld(d + unsigned(fl)) * (ct(1) - idx + fl) + dfrg::tld(d + unsigned(ceil(idx))) * (idx - fl);
    }

  private:
    static constexpr bool kLogFP64 = std::is_same_v<Coordinates, LogarithmicCoordinates1D<double>>;

    // the device index of FP64 log coordinates: sub-cell table and constants
    struct LogCells {
      const double2 *cell = nullptr; // {u_r, 1/(1 + u_r)} of sub-cell m = 0 .. K(N-1) - 1
      double c = 0, inv_b = 0;       // u = (x - c) inv_b; a NaN inv_b sends every point to the last one
      double s = 0, s_ln2 = 0;       // K(N-1)/a, K(N-1)/a ln 2
      double off = 0;                // o
      double inv_k = 1;              // 1/K
      double top = 0;                // N - 1
      int m_last = 0;                // last sub-cell (K(N-1) - 1)
      int last = 0;                  // last cell (N - 2; 0 for N = 1)
    };

    void make_cells()
    {
      const double a = coordinates.bias;
      const unsigned N = size;
      LogCells L;
      L.last = N >= 2 ? int(N) - 2 : 0;
      L.top = N - 1.;
      std::vector<double2> h;
      if (N >= 2 && a == a && a != 0) {
        if (!(std::fabs(a) <= 700.))
          throw std::invalid_argument("LinearInterpolator1D: the bias of LogarithmicCoordinates1D must be within "
                                      "[-700, 700] (exp(bias) overflows beyond)");
        int k_shift = 0;
        while (std::fabs(a) / ((double)(1u << k_shift) * (N - 1.)) > 1. / 32) ++k_shift;
        const double K = double(1u << k_shift), subs = K * (N - 1.);
        if (subs / std::fabs(a) * 0.69314718055994530942 > double(1 << 21) || subs > double(1 << 24))
          throw std::invalid_argument("LinearInterpolator1D: too many points for this bias of "
                                      "LogarithmicCoordinates1D (more than 2^21 sub-cells per unit of log2)");
        h.resize((size_t)subs);
        for (size_t m = 0; m < h.size(); ++m) {
          const double t = a * (double)(a > 0 ? m : m + 1) / subs, u = std::expm1(t);
          h[m] = make_double2(u, a > 0 ? 1. / (1. + u) : std::exp(-t));
        }
        L.c = coordinates.start;
        L.inv_b = 1. / ((coordinates.stop - coordinates.start) / std::expm1(a));
        L.s = subs / a;
        L.s_ln2 = subs / a * 0.69314718055994530942;
        L.off = a > 0 ? 0. : 1.;
        L.inv_k = 1. / K;
        L.m_last = int(subs) - 1;
      } else {
        // one point, bias 0 or NaN: the reference's index is 0 x (...)/a with a NaN or infinite
        // factor, or the one point; all points take the last point.  A valid dummy table keeps the
        // device code branch-free.
        h = {make_double2(0., 1.)};
        L.inv_b = std::numeric_limits<double>::quiet_NaN();
      }
      void *p = nullptr;
      dfrg::check(dfrg_malloc(&p, sizeof(double2) * h.size()), "LinearInterpolator1D cells");
      cells = std::shared_ptr<void>(p, [](void *q) { dfrg_free(q); });
      dfrg::check(dfrg_memcpy_h2d(p, h.data(), sizeof(double2) * h.size(), nullptr), "LinearInterpolator1D cells");
      dfrg::check(dfrg_stream_sync(nullptr), "LinearInterpolator1D cells");
      L.cell = (const double2 *)p;
      lc = L;
    }

    // the lerp at the reference's index of u = (x - c)/b (device, no branch on the grid)
    __device__ __forceinline__ NT log_cell_lerp(const double u_in) const
    {
      const double o = lc.off;
      const double off = u_in >= -1. ? o : 1e300; // 1e300: past the last point
      const double u = fmax(u_in, -1.);           // -1 for NaN
      // sub-cell estimate: log2(1 + u) = e + log2(mant), mant in [1/2, 1), FP32 log of the mantissa
      const double w = 1. + u;
      const double lg = (double)__builtin_amdgcn_logf((float)__builtin_amdgcn_frexp_mant(w));
      const double est = ((double)__builtin_amdgcn_frexp_exp(w) + lg) * lc.s_ln2;
      const int m = (int)fmax(0., fmin(est, (double)lc.m_last));
      const double2 cl = dfrg::gld(lc.cell + m); // {u_r, 1/(1 + u_r)}
      double dl = (u - cl.x) * cl.y;
      dl = fmax(-0.5, fmin(dl, 1.0)); // beyond the sub-cell by more than one: the clamp below decides
      double p = fma(dl, 0.13147226220077304, -0.16626609150418023);
      p = fma(p, dl, 0.1999935135656574);
      p = fma(p, dl, -0.24999995348000387);
      p = fma(p, dl, 0.3333333332203152);
      p = fma(p, dl, -0.4999999999999832);
      const double l = fma(dl * dl, p, dl); // log1p(dl)
      double idx = ((double)m + fma(lc.s, l, off)) * lc.inv_k;
      idx = fmax(0., fmin(idx, lc.top));
      const int i = min((int)idx, lc.last);
      const double f = idx - (double)i;
      const NT *d = device_data_ptr + i;
      return dfrg::gld(d) * (1. - f) + dfrg::gld(d + 1) * f;
    }

    unsigned size;
    Coordinates coordinates;
    std::shared_ptr<NT[]> m_data;
    std::shared_ptr<void> device_data;
    const NT *device_data_ptr = nullptr;
    bool owner;
    std::shared_ptr<void> cells;
    LogCells lc;
  };
} // namespace DiFfRG
