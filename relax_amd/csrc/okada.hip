// okada.hip -- Okada (1992) displacement of the shear patches and tensile
// cracks below the Nyquist size at the first event (relax.f90:357-360,
// dislocations_disp :1300-1349), on the device.
//
// grnfct_okada (okada/green_space.f90:119-146) evaluates, for every point
// of the half grid, Okada's closed-form displacement of a rectangular
// dislocation in a half-space (okada/dc3d.f, DC3D) and adds it to u.  Here
// one thread owns one grid point and walks the list of small sources in
// order, adding each one's displacement rounded to FP32 as the reference's
// REAL() does.  The closed form (Y. Okada, BSSA 82:1018-1040, Table 6) is
// evaluated in FP64 from single-precision arguments, as DC3D's REAL*4
// interface has them, with DC3D's treatment of singular points:
//  - |xi|, |eta|, |q| below 1e-6 count as 0;
//  - a point on a fault edge gives no displacement for that source;
//  - on the negative extension of an edge, ln(R + xi) becomes -ln(R - xi)
//    with X11 = X32 = 0 (likewise in eta);
//  - atan(xi eta / (q R)) is 0 for q = 0; |cos(dip)| < 1e-6 counts as 0.
#include <algorithm>
#include <cmath>
#include <vector>

#include "kernels.h"
#include "model.h"

namespace {

// One source in device form: the per-source constants of green_space.f90's
// okada() (its frame change and DC3D's single-precision arguments), formed
// on the host.
struct OkadaSource {
  double x1, x2;          // upper corner at the start of the strike (north, east)
  double csst, ssst;      // cos, sin of the strike
  double sd, cd, icd2;    // DC3D's dip constants (DCCON0), 1/cd^2
  float depth, al2, aw1;  // DEPTH, AL2 = length, AW1 = -width (AL1 = AW2 = 0)
  float d1, d2, d3;       // DISL1..3: slip cos(rake), slip sin(rake), opening
};

constexpr double OK_EPS = 1.0e-6;
constexpr double OK_PI2 = 6.283185307179586;

// Both sections of DC3D (the real source and its image) at one point need
// Table 6 at the four corners (xi, eta) of the fault, summed with the signs
// + - - + (Chinnery).  q, the dip and z are the same at the four corners, so
// the table is linear in a few corner sums and the transcendental terms
// collapse before they are evaluated:
//  - the signed sum of ln(R + eta) is one logarithm of a quotient of
//    products, likewise ln(R + xi) and ln(R + d~);
//  - the signed sum of four arc tangents is one atan2 of a product of complex
//    numbers: two of them lie within half a turn of each other, and the signs
//    of the pairs tell the full turns;
//  - roots and reciprocals are Newton steps on the hardware's estimates.
// The kernel is bound by FP64 issue: 129 sources on 256x256x64 points (541 M
// pairs) take 24.6 ms (about 900 FP64 instructions a pair, 214 VGPRs) against
// 103 ms with the table evaluated corner by corner (20 logarithms, 12 arc
// tangents, 18 roots and some 150 divisions a pair).  Held to 3 waves per
// SIMD (168 VGPRs, 50 spilled) it takes 36 ms, with the two sections in a loop
// 27 ms.
struct OkadaSums {
  double th, le, lx;               // th, ln(R+eta), ln(R+xi)
  double R1, X, Y, xY, eX;         // 1/R, X11, Y11, xi Y11, eta X11
  // the image only
  double lrd, at, xd, yd;          // ln(Rd), 2 atan of I4, xi/Rd, y~/Rd
  double ed, yd2, xyd2;            // vertical faults: eta/Rd, y~/Rd^2, xi y~/Rd^2
  double R3, eR3, eeR3;            // 1/R^3 and eta, eta^2 times it
  double X3, eX3, eeX3;            // X32 and eta, eta^2 times it
  double Z, xZ, xxZ;               // Z32 and xi, xi^2 times it
};

// 1/x from the hardware's estimate (better than 2^-26) and two Newton steps;
// x is normal here, so none of a division's scaling and special cases
__device__ __forceinline__ double ok_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}
// sqrt(x), x > 0, and 1/sqrt(x): Goldschmidt's iteration from the hardware's
// estimate
__device__ __forceinline__ double ok_root(double x, double& inv) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  inv = 2.0 * h;
  return g;
}
// a b and a - b rounded by themselves (no fused multiply-add)
__device__ __forceinline__ double ok_mul(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ double ok_sub(double a, double b) {
#pragma clang fp contract(off)
  return a - b;
}

// atan2(y0, x0) - atan2(y1, x1) with one atan2: the angle of the product of
// one number and the other's conjugate, a full turn apart where the
// difference leaves (-pi, pi)
__device__ __forceinline__ double ok_angle(double y0, double x0, double y1, double x1) {
  const double t = atan2(y0 * x1 - y1 * x0, x0 * x1 + y0 * y1);
  const double turn = (y0 >= 0.0 && y1 < 0.0 && t < 0.0) ? OK_PI2 : (y0 < 0.0 && y1 >= 0.0 && t > 0.0) ? -OK_PI2 : 0.0;
  return t + turn;
}

// The sums of one section.  kxi[k], ket[j] mark the negative extensions of the
// edges (k: eta corner, j: xi corner).
template <bool IMAGE>
__device__ __forceinline__ OkadaSums ok_sums(const double xi[2], const double et[2], double q, double z, double sd,
                                             double cd) {
  OkadaSums S{};
  double R[2][2], iR[2][2], re[2][2], rx[2][2], rd[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int k = 0; k < 2; ++k) R[j][k] = ok_root(xi[j] * xi[j] + et[k] * et[k] + q * q, iR[j][k]);
  const bool kxi[2] = {xi[0] < 0.0 && R[1][0] + xi[1] < OK_EPS, xi[0] < 0.0 && R[1][1] + xi[1] < OK_EPS};
  const bool ket[2] = {et[0] < 0.0 && R[0][1] + et[1] < OK_EPS, et[0] < 0.0 && R[1][1] + et[1] < OK_EPS};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    OkadaSums t[2];  // the terms of the two xi corners
    const double e = et[k];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const double x = xi[j];
      const double r = R[j][k], i1 = iR[j][k];
      // the logarithms' arguments, on an extension those of -ln(R - .)
      rx[j][k] = kxi[k] ? r - x : r + x;
      re[j][k] = ket[j] ? r - e : r + e;
      const double X11 = kxi[k] ? 0.0 : ok_mul(i1, ok_rcp(rx[j][k])), Y11 = ket[j] ? 0.0 : ok_mul(i1, ok_rcp(re[j][k]));
      t[j].R1 = i1;
      t[j].X = X11;
      t[j].Y = Y11;
      t[j].xY = x * Y11;
      if (IMAGE) {
        const double yt = e * cd + q * sd, d = r + (e * sd - q * cd), id = ok_rcp(d);
        rd[j][k] = d;
        t[j].xd = x * id;
        t[j].yd = ok_mul(yt, id);
        if (cd == 0.0) {
          t[j].ed = ok_mul(e, id);
          t[j].yd2 = ok_mul(yt * id, id);
          t[j].xyd2 = x * yt * id * id;
        }
        const double i3 = ok_mul(i1 * i1, i1), Y32 = (2.0 * r + e) * i1 * Y11 * Y11;
        t[j].R3 = i3;
        const double X32 = (2.0 * r + x) * i1 * X11 * X11;
        t[j].X3 = X32;
        const double Z32 = sd * i3 - (q * cd - z) * Y32;
        t[j].Z = Z32;
        t[j].xZ = x * Z32;
        t[j].xxZ = ok_mul(x * x, Z32);
      }
    }
    // a point midway along the strike has equal terms at the two corners:
    // their difference is exactly 0, as in the corner-by-corner sum
    const double sg = k == 0 ? 1.0 : -1.0;
#define OK_SUM(f) S.f += sg * ok_sub(t[0].f, t[1].f)
    OK_SUM(R1); OK_SUM(X); OK_SUM(Y); OK_SUM(xY); S.eX += sg * (e * ok_sub(t[0].X, t[1].X));
    if (IMAGE) {
      OK_SUM(xd); OK_SUM(yd);
      if (cd == 0.0) { OK_SUM(ed); OK_SUM(yd2); OK_SUM(xyd2); }
      const double r3 = sg * ok_sub(t[0].R3, t[1].R3), x3 = sg * ok_sub(t[0].X3, t[1].X3);
      S.R3 += r3; S.eR3 += e * r3; S.eeR3 += e * e * r3;
      S.X3 += x3; S.eX3 += e * x3; S.eeX3 += e * e * x3;
      OK_SUM(Z); OK_SUM(xZ); OK_SUM(xxZ);
    }
#undef OK_SUM
  }
  {
    double n = 1.0, d = 1.0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // + le(0,0) - le(0,1), - le(1,0) + le(1,1); reversed on an extension
      const double a = re[j][j], b = re[j][1 - j];
      n *= ket[j] ? b : a;
      d *= ket[j] ? a : b;
    }
    S.le = log(n / d);
  }
  {
    double n = 1.0, d = 1.0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double a = rx[k][k], b = rx[1 - k][k];
      n *= kxi[k] ? b : a;
      d *= kxi[k] ? a : b;
    }
    S.lx = log(n / d);
  }
  if (q != 0.0) {
    // the angles of the two xi corners, atan(p0/w0) - atan(p1/w1)
    const double aq = fabs(q);
    double y[2], w[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const double p0 = xi[j] * et[0], p1 = xi[j] * et[1], w0 = aq * R[j][0], w1 = aq * R[j][1];
      y[j] = p0 * w1 - p1 * w0;
      w[j] = w0 * w1 + p0 * p1;
    }
    const double t = ok_angle(y[0], w[0], y[1], w[1]);
    S.th = q < 0.0 ? -t : t;
  }
  if (IMAGE) {
    S.lrd = log((rd[0][0] * rd[1][1]) / (rd[0][1] * rd[1][0]));
    if (cd != 0.0) {
      double y[2], w[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        double i1;
        const double x = xi[j], X = ok_root(x * x + q * q, i1);
        const double r0 = R[j][0] + X, r1 = R[j][1] + X, c = fabs(x * cd);
        const double n0 = et[0] * (X + q * cd) + X * r0 * sd, n1 = et[1] * (X + q * cd) + X * r1 * sd;
        const double d0 = c * r0, d1 = c * r1, v = n0 * d1 - n1 * d0;
        y[j] = x * cd < 0.0 ? -v : v;
        w[j] = d0 * d1 + n0 * n1;
        if (x == 0.0) { y[j] = 0.0; w[j] = 1.0; }  // I4 = 0 there
      }
      S.at = 2.0 * ok_angle(y[0], w[0], y[1], w[1]);
    }
  }
  return S;
}

// DC3D's displacement at (X, Y, Z) (its single-precision arguments, widened);
// false at a singular point (on a fault edge).
__device__ __forceinline__ bool ok_dc3d(const OkadaSource& S, double alpha, double x, double y, double z, double u[3]) {
  const double sd = S.sd, cd = S.cd, c = S.depth;
  const double U1 = S.d1, U2 = S.d2, U3 = S.d3;
  u[0] = u[1] = u[2] = 0.0;
  const double a = alpha, b = 1.0 - alpha;
#pragma unroll
  for (int section = 0; section < 2; ++section) {
    double xi[2], et[2], q;
    {
      // the decisions below follow DC3D's own rounding
#pragma clang fp contract(off)
      xi[0] = x - 0.0;
      xi[1] = x - (double)S.al2;
      const double d = section == 0 ? c + z : c - z;
      const double p = y * cd + d * sd;
      q = y * sd - d * cd;
      et[0] = p - (double)S.aw1;
      et[1] = p - 0.0;
      if (fabs(q) < OK_EPS) q = 0.0;
      for (int k = 0; k < 2; ++k) {
        if (fabs(xi[k]) < OK_EPS) xi[k] = 0.0;
        if (fabs(et[k]) < OK_EPS) et[k] = 0.0;
      }
      if (q == 0.0 && ((xi[0] * xi[1] <= 0.0 && et[0] * et[1] == 0.0) || (et[0] * et[1] <= 0.0 && xi[0] * xi[1] == 0.0)))
        return false;
    }
    const OkadaSums T = section == 0 ? ok_sums<false>(xi, et, q, z, sd, cd) : ok_sums<true>(xi, et, q, z, sd, cd);
    const double q2 = q * q, a2 = a / 2, b2 = b / 2;
    // the A part (infinite medium): strike-slip, dip-slip and tensile rows
    double A0 = U1 * (T.th / 2 + a2 * q * T.xY) + U2 * (a2 * q * T.R1);
    double A1 = U1 * (a2 * q * T.R1) + U2 * (T.th / 2 + a2 * q * T.eX);
    double A2 = U1 * (b2 * T.le - a2 * q2 * T.Y) + U2 * (b2 * T.lx - a2 * q2 * T.X);
    if (U3 != 0.0) {
      A0 += U3 * (-b2 * T.le - a2 * q2 * T.Y);
      A1 += U3 * (-b2 * T.lx - a2 * q2 * T.X);
      A2 += U3 * (T.th / 2 - a2 * q * (T.eX + T.xY));
    }
    if (section == 0) {
      // the real source: -A (dc3d.f's real-source sum)
      u[0] = -A0;
      u[1] = -A1 * cd + A2 * sd;
      u[2] = -A1 * sd - A2 * cd;
      continue;
    }
    double I3, I4;
    if (cd != 0.0) {
      I4 = (T.xd * sd * cd + T.at) * S.icd2;
      I3 = (T.yd * cd - T.le + sd * T.lrd) * S.icd2;
    } else {
      I3 = (T.ed + q * T.yd2 - T.le) / 2.0;
      I4 = T.xyd2 / 2.0;
    }
    const double I1 = -T.xd * cd - I4 * sd, I2 = T.lrd + I3 * sd, k = b / a;
    double B0 = U1 * (-q * T.xY - T.th - k * I1 * sd) + U2 * (-q * T.R1 + k * I3 * sd * cd);
    double B1 = U1 * (-q * T.R1 + k * T.yd * sd) + U2 * (-q * T.eX - T.th - k * T.xd * sd * cd);
    double B2 = U1 * (q2 * T.Y - k * I2 * sd) + U2 * (q2 * T.X + k * I4 * sd * cd);
    // c~ = eta sin(dip) - h; y~ and d~ are linear in eta as well
    const double h = q * cd - z;
    const double yX = cd * T.eX + q * sd * T.X, dX = sd * T.eX - q * cd * T.X, cX = sd * T.eX - h * T.X;
    const double cR3 = sd * T.eR3 - h * T.R3, ceR3 = sd * T.eeR3 - h * T.eR3;
    const double cX3 = sd * T.eX3 - h * T.X3, ceX3 = sd * T.eeX3 - h * T.eX3;
    double C0 = U1 * (b * cd * T.xY - a * q * T.xZ) + U2 * (b * cd * T.R1 - q * sd * T.Y - a * q * cR3);
    double C1 = U1 * (b * (cd * T.R1 + 2.0 * q * sd * T.Y) - a * q * cR3) + U2 * (b * yX - a * q * ceX3);
    double C2 = U1 * (b * q * cd * T.Y - a * (ceR3 - z * T.Y + T.xxZ)) +
                U2 * (-dX - sd * T.xY - a * (cX - q2 * cX3));
    if (U3 != 0.0) {
      B0 += U3 * (q2 * T.Y - k * I3 * sd * sd);
      B1 += U3 * (q2 * T.X + k * T.xd * sd * sd);
      B2 += U3 * (q * (T.eX + T.xY) - T.th - k * I4 * sd * sd);
      C0 += U3 * (-b * (sd * T.R1 + q * cd * T.Y) - a * (z * T.Y - q2 * T.Z));
      C1 += U3 * (b * 2.0 * sd * T.xY + dX - a * (cX - q2 * cX3));
      C2 += U3 * (b * (yX + cd * T.xY) + a * q * (ceX3 + T.xZ));
    }
    // the image: A + B + z C, the vertical part of C reversed
    u[0] += A0 + B0 + z * C0;
    u[1] += (A1 + B1 + z * C1) * cd - (A2 + B2 + z * C2) * sd;
    u[2] += (A1 + B1 - z * C1) * sd + (A2 + B2 - z * C2) * cd;
  }
  for (int c3 = 0; c3 < 3; ++c3) u[c3] *= 1.0 / OK_PI2;
  return true;
}

// One thread per point of the h3 top planes of u (rows of ld floats, fields
// fs apart): the sources' displacements added in their order.
__global__ __launch_bounds__(256) void k_okada(const OkadaSource* __restrict__ src, int ns, float alpha, int n1,
                                               int n2, int h3, double dx1, double dx2, double dx3, float* u, long ld,
                                               long fs) {
#pragma clang fp contract(off)
  const long N = (long)n1 * n2 * h3;
  const long o = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (o >= N) return;
  const int i1 = o % n1, i2 = (o / n1) % n2, i3 = o / ((long)n1 * n2);
  // shiftedcoordinates (elastic3d.f90:4027-4048) and x3 = (i3-1) dx3
  const double xr = (double)(i1 < n1 / 2 ? i1 : i1 - n1) * dx1;
  const double yr = (double)(i2 < n2 / 2 ? i2 : i2 - n2) * dx2;
  const double zr = (double)i3 * dx3;
  const long of = i1 + ld * (i2 + (long)n2 * i3);
  float u1 = u[of], u2 = u[fs + of], u3 = u[2 * fs + of];
  const double Z = (double)(float)(-zr);
  for (int k = 0; k < ns; ++k) {
    const OkadaSource S = src[k];
    const double X = (double)(float)((xr - S.x1) * S.csst + (yr - S.x2) * S.ssst);
    const double Y = (double)(float)((xr - S.x1) * S.ssst - (yr - S.x2) * S.csst);
    double d[3];
    if (!ok_dc3d(S, (double)alpha, X, Y, Z, d)) continue;  // singular: no displacement
    const double UX = (double)(float)d[0], UY = (double)(float)d[1], UZ = (double)(float)d[2];
    u1 = u1 + (float)(UX * S.csst + UY * S.ssst);
    u2 = u2 + (float)(UX * S.ssst - UY * S.csst);
    u3 = u3 + (float)(-UZ);
  }
  u[of] = u1;
  u[fs + of] = u2;
  u[2 * fs + of] = u3;
}

}  // namespace

// The device form of a source given in the deck's convention (upper corner
// at the start of the strike, north-east-down, degrees), as green_space.f90's
// okada() derives DC3D's arguments from it.
static OkadaSource okada_source(double slip, double opening, const relax_source_t& s) {
  const double degtorad = (double)1.745329252e-2f;  // a single-precision literal (green_space.f90:47)
  OkadaSource S;
  S.x1 = s.x;
  S.x2 = s.y;
  const double st = s.strike * degtorad, ra = s.rake * degtorad;
  S.csst = std::cos(st);
  S.ssst = std::sin(st);
  // DCCON0: the dip in degrees as DC3D's single-precision argument
  const double dip = (double)(float)s.dip, p18 = 6.283185307179586 / 360.0;
  S.sd = std::sin(dip * p18);
  S.cd = std::cos(dip * p18);
  if (std::fabs(S.cd) < 1.0e-6) {
    S.cd = 0.0;
    S.sd = S.sd > 0.0 ? 1.0 : (S.sd < 0.0 ? -1.0 : S.sd);
  }
  S.icd2 = S.cd != 0.0 ? 1.0 / (S.cd * S.cd) : 0.0;
  S.depth = (float)s.z;
  S.al2 = (float)s.length;
  S.aw1 = -(float)s.width;
  S.d1 = (float)(slip * std::cos(ra));
  S.d2 = (float)(slip * std::sin(ra));
  S.d3 = (float)opening;
  return S;
}

// Launch over a padded or packed field set; the sources are staged in src
// (device memory of ns OkadaSource entries) from the host list hs.
static int launch_okada(const std::vector<OkadaSource>& hs, void* src, double lambda, double mu, int n1, int n2,
                        int h3, double dx1, double dx2, double dx3, float* u, long ld, long fs, hipStream_t st) {
  if (hs.empty()) return RELAX_OK;
  HIP_TRY(hipMemcpyAsync(src, hs.data(), sizeof(OkadaSource) * hs.size(), hipMemcpyHostToDevice, st));
  const float alpha = (float)((lambda + mu) / (lambda + 2.0 * mu));
  const long N = (long)n1 * n2 * h3;
  k_okada<<<(unsigned)((N + 255) / 256), 256, 0, st>>>((const OkadaSource*)src, (int)hs.size(), alpha, n1, n2, h3,
                                                      dx1, dx2, dx3, u, ld, fs);
  return hipGetLastError() == hipSuccess ? RELAX_OK : RELAX_ERR_HIP;
}

// dislocations_disp (relax.f90:1300-1349) on the model: the Okada
// displacement of the shear patches and tensile cracks at or below the
// nyquist size added to u, then sig = -tau + C:eps(u).
int relax_model_okada(relax_model_t* m, const relax_source_t* sc, int ns, const relax_source_t* tsc, int nt,
                      double nyquist) {
  if (!m || m->batch || ns < 0 || nt < 0 || (ns > 0 && !sc) || (nt > 0 && !tsc)) return RELAX_ERR_ARG;
  const double dmin = nyquist * std::min(m->desc.dx1, std::min(m->desc.dx2, m->desc.dx3));
  std::vector<OkadaSource> hs;
  for (int k = 0; k < ns; ++k)
    if (dmin >= sc[k].length || dmin >= sc[k].width) hs.push_back(okada_source(sc[k].slip, 0.0, sc[k]));
  for (int k = 0; k < nt; ++k)
    if (dmin >= tsc[k].length || dmin >= tsc[k].width) {
      relax_source_t t = tsc[k];
      t.rake = 0.0;
      hs.push_back(okada_source(0.0, tsc[k].opening, t));
    }
  if (hs.empty()) return RELAX_OK;
  void* src = nullptr;
  HIP_TRY(rx_malloc(&src, sizeof(OkadaSource) * hs.size()));
  const Grid& g = m->g;
  int rc = launch_okada(hs, src, m->desc.lambda, m->desc.mu, g.n1, g.n2, g.h3, m->desc.dx1, m->desc.dx2,
                        m->desc.dx3, m->u, g.n1, g.H, m->stream);
  if (!rc) rc = model_stress_set(m);
  if (hipStreamSynchronize(m->stream) != hipSuccess && !rc) rc = RELAX_ERR_HIP;
  (void)rx_free(src);
  return rc;
}

// grnfct_okada, okada/green_space.f90:119-146 (host arrays, added to)
int relax_grnfct_okada(double lambda, double mu, double slip, double opening, double x, double y, double z,
                       double width, double length, double strike, double dip, double rake, int sx1, int sx2, int sx3,
                       double dx1, double dx2, double dx3, float* u1, float* u2, float* u3, int align_data) {
  if (!u1 || !u2 || !u3 || sx1 < 1 || sx2 < 1 || sx3 < 1) return RELAX_ERR_ARG;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n < 1) return RELAX_ERR_NODEVICE;
  const long ld = align_data ? sx1 + 2 : sx1;
  const long fs = ld * sx2 * sx3;
  const relax_source_t s{slip, x, y, z, width, length, strike, dip, rake, 0.0, 0.0, 0.0, opening};
  std::vector<OkadaSource> hs{okada_source(slip, opening, s)};
  float* d = nullptr;
  void* src = nullptr;
  HIP_TRY(rx_malloc(&d, sizeof(float) * 3 * fs));
  int rc = rx_malloc(&src, sizeof(OkadaSource)) == hipSuccess ? RELAX_OK : RELAX_ERR_NOMEM;
  float* h[3] = {u1, u2, u3};
  for (int k = 0; k < 3 && !rc; ++k)
    if (hipMemcpy(d + k * fs, h[k], sizeof(float) * fs, hipMemcpyHostToDevice) != hipSuccess) rc = RELAX_ERR_HIP;
  if (!rc) rc = launch_okada(hs, src, lambda, mu, sx1, sx2, sx3, dx1, dx2, dx3, d, ld, fs, 0);
  if (!rc && rx_device_sync() != hipSuccess) rc = RELAX_ERR_HIP;
  for (int k = 0; k < 3 && !rc; ++k)
    if (hipMemcpy(h[k], d + k * fs, sizeof(float) * fs, hipMemcpyDeviceToHost) != hipSuccess) rc = RELAX_ERR_HIP;
  (void)rx_free(d);
  if (src) (void)rx_free(src);
  return rc;
}
