// The creep bands of rheology.h on the host: every grid point against the
// gates of frictioneigenstress (friction3d.f90:136-148), with and without
// fused multiply-adds, as a device compiler may form them.
#include <hip/hip_runtime.h>

#include <vector>

#include "model.h"
#include "rheology.h"

template <bool FUSED>
static bool gates(const RheoParams& R, const PlaneDev& P, int i1, int i2, int i3) {
#pragma clang fp contract(off)
  const double f1 = (double)(i1 < R.n1 / 2 ? i1 : i1 - R.n1), f2 = (double)(i2 < R.n2 / 2 ? i2 : i2 - R.n2), f3 = (double)i3;
  const double x1 = f1 * R.dx1, x2 = f2 * R.dx2, x3 = f3 * R.dx3;
  auto minus = [](double a, double d, double b) { return FUSED ? fma(a, d, -b) : a * d - b; };
  const double wl = fmax(P.Wp, P.Lp);
  if (fabs(minus(f3, R.dx3, P.z)) > P.Lp && fabs(minus(f3, R.dx3, -P.z)) > P.Lp) return false;
  if (fabs(minus(f1, R.dx1, P.x)) > wl || fabs(minus(f2, R.dx2, P.y)) > wl) return false;
  const double c = FUSED ? fma(P.cstrike, x1, -(P.sstrike * x2)) : P.cstrike * x1 - P.sstrike * x2;
  const double s = FUSED ? fma(P.cdip, c, -(P.sdip * x3)) : P.cdip * c - P.sdip * x3;
  const double i = FUSED ? fma(P.cdip, c, P.sdip * x3) : P.cdip * c + P.sdip * x3;
  return !(fabs(s - P.xr) > 7.01 * R.dx1 && fabs(i - P.xr) > 7.01 * R.dx1);
}

static void setup(const relax_plane_t* planes, int np, double beta, const int* n, const double* dx, RheoParams& R,
                  std::vector<PlaneDev>& P) {
  for (int k = 0; k < np; ++k) P.push_back(make_plane(planes[k], beta, dx[0], dx[2]));
  R.n1 = n[0]; R.n2 = n[1];
  R.dx1 = dx[0]; R.dx2 = dx[1]; R.dx3 = dx[2];
  R.fr.planes = P.data();
  R.fr.np = np;
  band_box(R.fr, P.data(), np, n[0], n[1], n[2], dx[0], dx[1], dx[2]);
}

// box: zmax, x0, nx, y0, ny
extern "C" void creep_box(const relax_plane_t* planes, int np, double beta, const int* n, const double* dx, int* box) {
  RheoParams R{};
  std::vector<PlaneDev> P;
  setup(planes, np, beta, n, dx, R, P);
  const int b[5] = {R.fr.zmax, R.fr.x0, R.fr.nx, R.fr.y0, R.fr.ny};
  for (int k = 0; k < 5; ++k) box[k] = b[k];
}

// out: points within the gates, those of them outside the band, outside their
// column's range, outside the box; and columns with a range outside the box
extern "C" void creep_sweep(const relax_plane_t* planes, int np, double beta, const int* n, const double* dx, long* out) {
  RheoParams R{};
  std::vector<PlaneDev> P;
  setup(planes, np, beta, n, dx, R, P);
  const FrictionTables& F = R.fr;
  for (int k = 0; k < 5; ++k) out[k] = 0;
  for (int i2 = 0; i2 < n[1]; ++i2)
    for (int i1 = 0; i1 < n[0]; ++i1) {
      int lo, hi;
      column_band(R, i1, i2, lo, hi);
      const bool box = (i1 - F.x0 + n[0]) % n[0] < F.nx && (i2 - F.y0 + n[1]) % n[1] < F.ny;
      if (lo <= hi && (!box || hi >= F.zmax)) ++out[4];
      for (int i3 = 0; i3 < n[2]; ++i3) {
        bool g = false;
        for (int k = 0; k < np; ++k) g = g || gates<false>(R, P[k], i1, i2, i3) || gates<true>(R, P[k], i1, i2, i3);
        if (!g) continue;
        ++out[0];
        if (!in_band(R, i1, i2, i3)) ++out[1];
        if (i3 < lo || i3 > hi) ++out[2];
        if (!box || i3 >= F.zmax) ++out[3];
      }
    }
}
