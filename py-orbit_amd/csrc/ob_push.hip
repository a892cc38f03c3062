// ob_push.hip -- the fused TEAPOT map kernel.
//
// One launch applies a program of queued maps (drift, quad1, quad2, quad/multipole
// fringes, multipole kicks, wraps, rotations, plain kicks) and the deferred
// space-charge kicks to every particle, holding the six FP64 coordinates in
// registers: each particle is read once and written once per launch (96 B) however
// many maps the program holds.  When the program feeds a space-charge node it also
// emits per-block min/max of x, y, z for the next grid (BunchExtremaCalculator.cc:
// 37-83), so the extrema pass costs no extra HBM read.
//
// Arithmetic follows the reference routine of each map operation for operation
// (cited per case), compiled with -ffp-contract=off so nothing is fused: results
// are bit-identical to src/teapot/teapotbase.cc built with g++ for x86-64.
#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "ob_internal.hpp"
#include "ob_sc_device.hpp"
#include "ob_tiled3d.hpp"
#include "ob_tiled3d_device.hpp"

namespace ob {

namespace {

struct cplx {
  double re, im;
};
__device__ __forceinline__ cplx cmul(cplx a, cplx b) {  // std::complex<double> product
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }

// teapotbase.cc:395-490 / 508-603.  kk = (kre, kim) = +/-kterm, pole; the reference's complex
// products by real or imaginary constants (l, l + 2, i) without their zero terms, which add
// +-0 to finite values: the same results, a third fewer operations.
__device__ __forceinline__ void multpfringe(int pole, double kre, double kim, double KNL,
                                            double& x, double& xp, double& y, double& yp,
                                            double& z) {
  const double l = (double)(pole + 1), lp2 = (double)(pole + 3);
  const double px = xp, py = yp;
  const cplx zz = {x, y};
  cplx zlm1 = {1.0, 0.0};
  if (pole > 0) zlm1 = zz;
  for (int k = 1; k < pole; k++) zlm1 = cmul(zlm1, zz);
  const cplx zl = pole > 0 ? cmul(zlm1, zz) : zz;
  const cplx fxterm = {l * x, -lp2 * y};
  const cplx fxz = cadd(fxterm, zz);
  const cplx dxfxterm = {l * fxz.re, l * fxz.im};
  const cplx w = {l * fxterm.re - lp2 * zz.re, l * fxterm.im - lp2 * zz.im};
  const cplx dyfxterm = {-w.im, w.re};
  const cplx fyterm = {l * y, lp2 * x};
  const cplx dxfyterm = {l * fyterm.re - lp2 * zz.im, l * fyterm.im + lp2 * zz.re};
  const cplx ify = {-fyterm.im + zz.re, fyterm.re + zz.im};
  const cplx dyfyterm = {l * ify.re, l * ify.im};
  cplx kzl, kzlm1;
  if (kim == 0.0) {  // uniform: a normal multipole's coefficient is real
    kzl = {kre * zl.re, kre * zl.im};
    kzlm1 = {kre * zlm1.re, kre * zlm1.im};
  } else {
    const cplx kk = {kre, kim};
    kzl = cmul(kk, zl);
    kzlm1 = cmul(kk, zlm1);
  }
  const cplx fxcx = cmul(kzl, fxterm);
  const cplx dxfxcx = cmul(kzlm1, dxfxterm);
  const cplx dyfxcx = cmul(kzlm1, dyfxterm);
  const cplx fycx = cmul(kzl, fyterm);
  const cplx dxfycx = cmul(kzlm1, dxfyterm);
  const cplx dyfycx = cmul(kzlm1, dyfyterm);
  x -= fxcx.re * KNL;
  y -= fycx.re * KNL;
  const double M11 = 1.0 - dxfxcx.re * KNL;
  const double M12 = -dxfycx.re * KNL;
  const double M21 = -dyfxcx.re * KNL;
  const double M22 = 1.0 - dyfycx.re * KNL;
  const double detM = M11 * M22 - M12 * M21;
  const double pxnew = (M22 * px - M12 * py) / detM;
  const double pynew = (-M21 * px + M11 * py) / detM;
  xp = pxnew;
  yp = pynew;
  z -= (pxnew * fxcx.re + pynew * fycx.re) * KNL * KNL;
}

// teapotbase.cc:784-835 (IN) / 854-905 (OUT).
__device__ __forceinline__ void quadfringe(bool out, double kq, double KNL, double& x, double& xp,
                                           double& y, double& yp, double& z) {
  const double x0 = x, xp0 = xp, y0 = y, yp0 = yp;
  const double t = (kq * KNL / 4.) * (x0 * x0 - y0 * y0);
  const double detM = 1.0 - t * t;
  double dx = (kq * KNL / 12.) * x0 * (x0 * x0 + 3. * y0 * y0);
  double dxp = (kq * KNL / 4.) * (xp0 * (x0 * x0 + y0 * y0) - 2. * yp0 * x0 * y0);
  double dy = (kq * KNL / 12.) * y0 * (y0 * y0 + 3. * x0 * x0);
  double dyp = (kq * KNL / 4.) * (-yp0 * (x0 * x0 + y0 * y0) + 2. * xp0 * x0 * y0);
  double dz = (kq * KNL * KNL / 12.) *
              (xp0 * x0 * (x0 * x0 + 3. * y0 * y0) - yp0 * y0 * (y0 * y0 + 3. * x0 * x0));
  if (out) {  // uniform; a - b and a + (-b) are the same value
    dx = -dx;
    dxp = -dxp;
    dy = -dy;
    dyp = -dyp;
    dz = -dz;
  }
  x += dx;
  xp -= dxp;
  xp /= detM;
  y -= dy;
  yp -= dyp;
  yp /= detM;
  z += dz;
}

// One particle's drift (drifti, teapotbase.cc:120-141).
__device__ __forceinline__ void drift_one(double length, double gamma2i, double dp_p, double KNL,
                                          double& x, double xp, double& y, double yp,
                                          double& z) {
  x += KNL * length * xp;
  y += KNL * length * yp;
  double phifac = (xp * xp + yp * yp + dp_p * dp_p * gamma2i) / 2.0;
  phifac = (phifac * KNL - dp_p * gamma2i) * KNL;
  z -= length * phifac;
}

// wedgebend / wedgebendCF (teapotbase.cc:1037-1080, 1447-1509).  w: ct, rho, poles (4 bits
// each, low half) and nst, then kl of the nm multipoles; ia = inout | nm << 1 | skew bits << 8.
// The multipole kick of each step is multpi (:280-315) with kl * sm, divided by pole! per particle
// as there.
template <typename W>
__device__ __forceinline__ void wedgebend(W w, uint32_t ia, double gamma2i, double dp_p,
                                          double KNL, double& x, double& xp, double& y,
                                          double& yp, double& z) {
  const double ct = w[0], rho = w[1];
  const uint64_t pn = (uint64_t)__double_as_longlong(w[2]);
  const uint32_t poles = (uint32_t)pn;
  const int inout = ia & 1, nm = (ia >> 1) & 15, skews = (ia >> 8) & 255;
  const int nst = (int)(pn >> 32);
  double s;
  if (inout == 0) {
    s = -x / ct;
  } else {
    const double tn = xp / (1.0 + dp_p);
    s = -x / (ct + tn);
  }
  const double sm = s / nst, sm2 = sm / 2.0;
  for (int j = 0; j < nst; j++) {
    drift_one(j == 0 ? sm2 : sm, gamma2i, dp_p, KNL, x, xp, y, yp, z);
    xp -= sm / rho;
    for (int l = 0; l < nm; l++) {
      const int pole = (poles >> (4 * l)) & 15;
      double fact = 1.0;  // teapotbase.cc:45-57
      for (int k = 1; k <= pole; k++) fact = k * fact;
      const double kl1 = (w[3 + l] * sm) / fact;
      const cplx zz = {x, y};
      cplx zn = {1.0, 0.0};
      for (int k = 0; k < pole; k++) zn = cmul(zn, zz);
      if ((skews >> l) & 1) {
        xp += kl1 * zn.im;
        yp += kl1 * zn.re;
      } else {
        xp -= kl1 * zn.re;
        yp += kl1 * zn.im;
      }
    }
  }
  drift_one(sm2, gamma2i, dp_p, KNL, x, xp, y, yp, z);
}

// soln (teapotbase.cc:1367-1425).
__device__ __forceinline__ void soln(double Bc, double length, double gamma2i, double dp_p,
                                     double KNL, double& x, double& xp, double& y, double& yp,
                                     double& z) {
  const double cu = y / 2. - xp / Bc;
  const double cpu = x * Bc / 2. + yp;
  const double u_init = y / 2. + xp / Bc;
  const double pu_init = -x * Bc / 2. + yp;
  const double phase = KNL * Bc * length;
  const double cs = cos(phase), sn = sin(phase);
  const double u = u_init * cs + pu_init * sn / Bc;
  const double pu = -u_init * Bc * sn + pu_init * cs;
  x = (-pu + cpu) / Bc;
  xp = 0.5 * (u - cu) * Bc;
  y = u + cu;
  yp = 0.5 * (pu + cpu);
  double phifac = (pu_init * pu_init + Bc * Bc * u_init * u_init + dp_p * dp_p * gamma2i) / 2.0;
  phifac = (phifac * KNL - dp_p * gamma2i) * KNL;
  z -= length * phifac;
}

// Kernel level an op kind needs: 0 = the lite kernels, 1 = with the multipole fringes (a
// ring's sextupoles), 2 = with wedge bend, solenoid and ring RF, 3 = with space-charge kicks
// inside a program (a calculator's kick leads its queue: 2.5D kicks run before the program, 3D
// ones outside the deposit's tiles take this level).  Each level holds the ones below it; a
// lower level runs with fewer VGPRs and so more waves per SIMD (maps only: 62, 70, 100, 214).
constexpr int kLevels = 4;
__host__ __device__ constexpr int op_level(int kind) {
  return (kind == OP_MULTPFRINGE_IN || kind == OP_MULTPFRINGE_OUT) ? 1
         : (kind == OP_WEDGEBEND || kind == OP_SOLN || kind == OP_RINGRF) ? 2
         : (kind == OP_SC2P5DRB_KICK || kind == OP_SC3D_KICK) ? 3
                                                               : 0;
}

// The whole program (ProgramWords) on one particle.  The next op's header is requested before
// this op runs (all lanes run the same op: the words are scalar loads).
template <int LEVEL, typename PROG>
__device__ __forceinline__ void run_program(const PROG& prog, double& x, double& xp, double& y,
                                            double& yp, double& z, double& dE) {
  double dpc = prog.dpc, g2i = prog.g2i;
  double dp_p = 0.0, KNL = 0.0;
  const int words = prog.words;
  uint64_t hdr = words > 0 ? (uint64_t)__double_as_longlong(prog.data[0]) : 0;
  for (int pc = 0; pc < words;) {
    const uint32_t h = (uint32_t)hdr, ia = (uint32_t)(hdr >> 32);
    const double* w = prog.data + pc + 1;
    pc += (int)((h >> 12) & 255u);
    hdr = (uint64_t)__double_as_longlong(prog.data[pc < words ? pc : 0]);
    if (h & kProgRecalc) {
      dp_p = dE * dpc;
      KNL = 1.0 / (1.0 + dp_p);
    }
    switch (h & 255u) {
      case OP_DRIFT:  // teapotbase.cc:158-183.  length
        drift_one(w[0], g2i, dp_p, KNL, x, xp, y, yp, z);
        break;
      case OP_QUAD1: {  // teapotbase.cc:686-699.  m11 = m22, m12, m21, m33 = m44, m34, m43, length
        const double x0 = x, xp0 = xp, y0 = y, yp0 = yp;
        x = x0 * w[0] + xp0 * w[1];
        xp = x0 * w[2] + xp0 * w[0];
        y = y0 * w[3] + yp0 * w[4];
        yp = y0 * w[5] + yp0 * w[3];
        z += dp_p * g2i * w[6];
        break;
      }
      case OP_QUAD2: {  // teapotbase.cc:719-745.  length
        const double length = w[0];
        x -= KNL * length * dp_p * xp;
        y -= KNL * length * dp_p * yp;
        double phifac = (xp * xp + yp * yp + dp_p * dp_p * g2i) / 2.0;
        phifac = (phifac * KNL + dp_p * dp_p * g2i) * KNL;
        z -= length * phifac;
        break;
      }
      case OP_QUADFRINGE_IN:   // kq
      case OP_QUADFRINGE_OUT:
        quadfringe((h & 255u) == OP_QUADFRINGE_OUT, w[0], KNL, x, xp, y, yp, z);
        break;
      case OP_MULTP: {  // teapotbase.cc:336-372.  kl/pole!; ia = pole | skew << 8
        const cplx zz = {x, y};
        cplx zn = {1.0, 0.0};
        const int pole = (int)(ia & 255u);
        for (int k = 0; k < pole; k++) zn = cmul(zn, zz);
        const double kl1 = w[0];
        if (ia >> 8) {
          xp += kl1 * zn.im;
          yp += kl1 * zn.re;
        } else {
          xp -= kl1 * zn.re;
          yp += kl1 * zn.im;
        }
        break;
      }
      case OP_MULTPFRINGE_IN:
      case OP_MULTPFRINGE_OUT:  // kre, kim; ia = pole
        if constexpr (LEVEL >= 1) multpfringe((int)ia, w[0], w[1], KNL, x, xp, y, yp, z);
        break;
      case OP_WRAPBUNCH: {  // teapotbase.cc:202-211.  length
        const double length = w[0];
        if (z < -length / 2.0) z += length;
        if (z > length / 2.0) z -= length;
        break;
      }
      case OP_ROTATEXY: {  // teapotbase.cc:80-101.  cos, sin
        const double cs = w[0], sn = w[1];
        const double xt = x, pxt = xp, yt = y, pyt = yp;
        x = cs * xt - sn * yt;
        xp = cs * pxt - sn * pyt;
        y = sn * xt + cs * yt;
        yp = sn * pxt + cs * pyt;
        break;
      }
      case OP_KICK:  // teapotbase.cc:232-257.  kx, ky, kE
        if (w[0] != 0.) xp += w[0];
        if (w[1] != 0.) yp += w[1];
        if (w[2] != 0.) dE += w[2];
        break;
      case OP_SC2P5DRB_KICK:  // p[0..5]; ia = nx, then a word with ny, nz
        if constexpr (LEVEL >= 3) sc2p5drb_kick(w, (int)ia, x, xp, y, yp, z, dE);
        break;
      case OP_SC3D_KICK:  // p[0..11]; ia = nx, then a word with ny, nz
        if constexpr (LEVEL >= 3) sc3d_kick(w, (int)ia, x, xp, y, yp, z, dE);
        break;
      case OP_BEND1: {  // teapotbase.cc:1099-1145.  m11 m12 m16 m21 m22 m26 m51 m52 m56, length
        const double x0 = x, xp0 = xp;
        x = x0 * w[0] + xp0 * w[1] + dp_p * w[2];
        xp = x0 * w[3] + xp0 * w[4] + dp_p * w[5];
        y += w[9] * yp;
        z += x0 * w[6] + xp0 * w[7] + dp_p * w[8];
        break;
      }
      case OP_BEND3: {  // teapotbase.cc:1208-1233.  th
        const double th = w[0];
        double phifac = (yp * yp + dp_p * dp_p * g2i) / 2.0;
        xp -= phifac * KNL * th;
        y += KNL * yp * x * th;
        phifac = (phifac * KNL - dp_p * g2i) * KNL;
        z -= th * phifac * x;
        break;
      }
      case OP_BEND4: {  // teapotbase.cc:1251-1274.  th
        const double th = w[0];
        const double xfac = 1.0 + KNL * xp * th / 2.0;
        const double phifac = KNL * KNL * xp * xp / 2.0;
        x *= xfac * xfac;
        xp /= xfac;
        z -= th * phifac * x;
        break;
      }
      case OP_BENDFRINGE_IN:     // teapotbase.cc:1292-1311.  rho
      case OP_BENDFRINGE_OUT: {  // teapotbase.cc:1329-1348
        const double rho = w[0];
        if ((h & 255u) == OP_BENDFRINGE_IN) {
          x += KNL * y * y / (2. * rho);
          yp -= KNL * xp * y / rho;
          z += KNL * KNL * xp * y * y / (2. * rho);
        } else {
          x -= KNL * y * y / (2. * rho);
          yp += KNL * xp * y / rho;
          z -= KNL * KNL * xp * y * y / (2. * rho);
        }
        break;
      }
      case OP_WEDGEROTATE: {  // teapotbase.cc:923-966.  cos e, sin e; ia = frinout
        const double cs = w[0], sn = w[1];
        double dp, xp_temp, p0_temp, p0;
        if (ia == 0) {
          dp = dE * dpc;
          xp_temp = xp;
          p0_temp = 1.0 + dp;
          x /= cs;
          xp = xp_temp * cs + p0_temp * sn;
          p0 = -xp_temp * sn + p0_temp * cs;
          dp = p0 - 1.0;
          z = (-x * sn + z) * cs;
        } else {
          dp = dE * dpc;
          p0 = 1.0 + dp;
          z = x * sn + z / cs;
          x *= cs;
          xp_temp = xp * cs - p0 * sn;
          p0_temp = xp * sn + p0 * cs;
          xp = xp_temp;
          dp = p0_temp - 1.0;
        }
        dE = dp / dpc;
        break;
      }
      case OP_WEDGEDRIFT: {  // teapotbase.cc:986-1012.  ct; ia = inout
        const double ct = w[0];
        double s;
        if (ia == 0) {
          const double tn = xp / (1.0 + dp_p);
          s = x / (ct - tn);
        } else {
          s = x / ct;
        }
        drift_one(s, g2i, dp_p, KNL, x, xp, y, yp, z);
        break;
      }
      case OP_WEDGEBEND:
        if constexpr (LEVEL >= 2) wedgebend(w, ia, g2i, dp_p, KNL, x, xp, y, yp, z);
        break;
      case OP_SOLN:  // Bc, length
        if constexpr (LEVEL >= 2) soln(w[0], w[1], g2i, dp_p, KNL, x, xp, y, yp, z);
        break;
      case OP_RINGRF:  // teapotbase.cc:1527-1566.  h*2pi/L, phase_s, voltage, coeff, p_in/p_out
        if constexpr (LEVEL >= 2) {
          const double deltaV = w[2] * (sin(w[0] * z + w[1]));
          dE += w[3] * deltaV;
          xp *= w[4];
          yp *= w[4];
        }
        break;
      case OP_ENV:
        dpc = w[0];
        g2i = w[1];
        break;
      default:
        break;
    }
  }
}

constexpr int kPushThreads = 256;
constexpr int kMaxPushBlocks = 4096;
constexpr int kKickPushBlocks = 1024;

__device__ __forceinline__ double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Extrema of a workgroup's x, y, z (each thread's in lo, hi) to its row of partials.
__device__ __forceinline__ void block_extrema(const double lo[3], const double hi[3],
                                              double* __restrict__ partials) {
  __shared__ double red[kPushThreads / 64][6];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double r[6];
  for (int k = 0; k < 3; k++) {
    r[2 * k] = wave_min(lo[k]);
    r[2 * k + 1] = wave_max(hi[k]);
  }
  if (lane == 0)
    for (int k = 0; k < 6; k++) red[w][k] = r[k];
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    double acc = red[0][k];
    for (int j = 1; j < kPushThreads / 64; j++)
      acc = (k & 1) ? fmax(acc, red[j][k]) : fmin(acc, red[j][k]);
    partials[(int64_t)blockIdx.x * 6 + k] = acc;
  }
}

template <typename P>
__device__ __forceinline__ void load6(P a, P b, P c, P d, P e, P f, int64_t i, double q[6]) {
  q[0] = a[i];
  q[1] = b[i];
  q[2] = c[i];
  q[3] = d[i];
  q[4] = e[i];
  q[5] = f[i];
}

// KICK0: a SpaceChargeCalc2p5Drb kick comes before the program (the usual case: the deferred
// kick of the previous SC node); it runs outside the op interpreter, with the calculator's
// values read once, before any store (scalar loads).  Without it the kernel keeps the
// interpreter's smaller register footprint.  W: the program's words in the kernel arguments; a
// step's few maps take the small form, since every launch copies its arguments on the host
// (2.7 KB 0.9 us more than a few hundred bytes).
struct Kick0 {
  const SC2DState* st;
  const double *phi, *zg, *zd;
  double p4, p5;
  int32_t nx, ny, nz, pad;
};
template <bool EXTREMA, int LEVEL, bool KICK0, int W>
__global__ __launch_bounds__(kPushThreads) void push_kernel(DeviceBunchView v,
                                                            ProgramWords<W> prog, Kick0 k0,
                                                            double* __restrict__ partials) {
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
  double hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const gptr<double> cx = to_global(v.c[0]);
  const gptr<double> cxp = to_global(v.c[1]);
  const gptr<double> cy = to_global(v.c[2]);
  const gptr<double> cyp = to_global(v.c[3]);
  const gptr<double> cz = to_global(v.c[4]);
  const gptr<double> cdE = to_global(v.c[5]);
  SC2DKickParams kp;
  if constexpr (KICK0) kp = sc2d_kick_params(k0.st);
  // The next particle's coordinates are loaded before this one is computed (after its
  // kick's loads), so their latency overlaps the kick and map arithmetic (few waves fit:
  // the map switch needs many VGPRs).
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double q[6];
  if (i < v.n) load6(cx, cxp, cy, cyp, cz, cdE, i, q);
  for (; i < v.n; i += stride) {
    double x = q[0], xp = q[1], y = q[2], yp = q[3], z = q[4], dE = q[5];
    SC2DKickLoads L;
    if constexpr (KICK0)
      sc2p5drb_kick_loads(kp, to_global(k0.phi), k0.nx, k0.ny, to_global(k0.zg),
                          to_global(k0.zd), k0.nz, x, y, z, L);
    if (i + stride < v.n) load6(cx, cxp, cy, cyp, cz, cdE, i + stride, q);
    if constexpr (KICK0) sc2p5drb_kick_apply(kp, L, k0.nz, k0.p4, k0.p5, x, xp, y, yp, dE);
    run_program<LEVEL>(prog, x, xp, y, yp, z, dE);
    cx[i] = x;
    cxp[i] = xp;
    cy[i] = y;
    cyp[i] = yp;
    cz[i] = z;
    cdE[i] = dE;
    if (EXTREMA) {
      lo[0] = fmin(lo[0], x);
      hi[0] = fmax(hi[0], x);
      lo[1] = fmin(lo[1], y);
      hi[1] = fmax(hi[1], y);
      lo[2] = fmin(lo[2], z);
      hi[2] = fmax(hi[2], z);
    }
  }
  if (EXTREMA) block_extrema(lo, hi, partials);
}

// The kick of a tile-sorted bunch (ob_tiled3d.hip) and the program of the maps after it, one pass
// over the particles.  Workgroups walk the work items: a tile's block of phi goes to LDS, its
// particles are kicked from it; item nitems is the particles outside the grid (last in the
// sorted order, from offsets[ntiles]), kicked from the whole grid like the reference.  MAPS:
// false without a program and extrema (three of the six coordinates are written).
// As two launches the kick and the push moved 72 + 96 bytes per particle; here 96.
// At least 3 waves per SIMD: the kick with the next particle's prefetch takes 157 VGPRs
// without spills.  Bounded to 4 waves (128 VGPRs) the prefetch spills and the kick ran
// 133 us against 113; without the prefetch, 119.
template <bool BND, bool EXTREMA, int LEVEL, bool MAPS>
__global__ __launch_bounds__(kTileThreads, 3) void tile_push(
    double* __restrict__ cur, int64_t cap, TileKick t, ProgramWords<kProgSmallWords> prog,
    double* __restrict__ partials) {
  const TileGeom& g = t.g;
  const Kick3D& k = t.k;
  const uint32_t ni = *t.nitems;
  extern __shared__ double sphi[];
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
  double hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  auto finish = [&](int64_t i, double x, double xp, double y, double yp, double z, double dE) {
    if constexpr (MAPS) {
      run_program<LEVEL>(prog, x, xp, y, yp, z, dE);
      cur[i] = x;
      cur[2 * cap + i] = y;
      cur[4 * cap + i] = z;
    }
    cur[cap + i] = xp;
    cur[3 * cap + i] = yp;
    cur[5 * cap + i] = dE;
    if constexpr (EXTREMA) {
      lo[0] = fmin(lo[0], x);
      hi[0] = fmax(hi[0], x);
      lo[1] = fmin(lo[1], y);
      hi[1] = fmax(hi[1], y);
      lo[2] = fmin(lo[2], z);
      hi[2] = fmax(hi[2], z);
    }
  };
  const int64_t gsx = (int64_t)g.ny * g.nz;
  for (uint32_t item = blockIdx.x; item <= ni; item += gridDim.x) {
    const bool rest = item == ni;
    const int4 it = rest ? make_int4(0, (int)t.offsets[g.ntiles], (int)t.n, 0) : t.items[item];
    TileBox box(g, it.x);
    if (rest) box.x0 = 1 << 30;  // no block: holds no node
    const int cells = box.cells();
    // The first particle's coordinates are requested with the block of phi, and all of a
    // thread's block loads are issued before any is stored (a masked lane loads phi[0] and
    // stores 0), so these latencies overlap instead of adding up.
    const int i0 = it.y + (int)threadIdx.x;
    const int ia = i0 < it.z ? i0 : 0;
    double q[6] = {cur[ia], cur[2 * cap + ia], cur[4 * cap + ia],
                   cur[cap + ia], cur[3 * cap + ia], cur[5 * cap + ia]};
    constexpr int KB = 8;  // cells <= KB * kTileThreads for blocks of up to 16 KiB
    double bv[KB];
    uint32_t inmask = 0;
    CellWalk w((int)threadIdx.x, box.W, box.Wz);
#pragma unroll
    for (int u = 0; u < KB; u++, w.next()) {
      const int c = (int)threadIdx.x + u * kTileThreads;
      const int gx = box.x0 + w.lx, gy = box.y0 + w.ly, gz = box.z0 + w.lz;
      const bool in = c < cells && gx >= 0 && gx < g.nx && gy >= 0 && gy < g.ny && gz >= 0 &&
                      gz < g.nz;
      bv[u] = k.phi[in ? gx * gsx + (int64_t)gy * g.nz + gz : 0];
      inmask |= (in ? 1u : 0u) << u;
    }
    if (item != blockIdx.x) __syncthreads();  // the last item's block is no longer read
#pragma unroll
    for (int u = 0; u < KB; u++) {
      const int c = (int)threadIdx.x + u * kTileThreads;
      if (c < cells) sphi[c] = ((inmask >> u) & 1u) ? bv[u] : 0.0;
    }
    for (int c = (int)threadIdx.x + KB * kTileThreads; c < cells; c += kTileThreads, w.next()) {
      // larger blocks: the walk continues from cell threadIdx.x + KB * kTileThreads
      const int gx = box.x0 + w.lx, gy = box.y0 + w.ly, gz = box.z0 + w.lz;
      const bool in = gx >= 0 && gx < g.nx && gy >= 0 && gy < g.ny && gz >= 0 && gz < g.nz;
      sphi[c] = in ? k.phi[gx * gsx + (int64_t)gy * g.nz + gz] : 0.0;
    }
    __syncthreads();
    // The next particle's coordinates are loaded before this one is kicked.
    for (int i = i0; i < it.z; i += kTileThreads) {
      const int in = i + kTileThreads < it.z ? i + kTileThreads : i;
      const double nq[6] = {cur[in], cur[2 * cap + in], cur[4 * cap + in],
                            cur[cap + in], cur[3 * cap + in], cur[5 * cap + in]};
      tile_kick_particle<BND>(g, k, sphi, box, q[0], q[1], q[2], q[3], q[4], q[5]);
      finish(i, q[0], q[3], q[1], q[4], q[2], q[5]);
#pragma unroll
      for (int c = 0; c < 6; c++) q[c] = nq[c];
    }
  }
  if constexpr (EXTREMA) block_extrema(lo, hi, partials);
}

// Potentials of at most this many nodes (64 x 64) are copied into LDS by each workgroup
// of the batch push: the kick's nine gathers per particle then read LDS, where 64
// random addresses cost a few cycles, instead of the L1/L2 path, where they cost a
// cache-line lookup per lane.
constexpr int kBatchPhiLds = 4096;

// All bunches of a batch in one launch: block = one work item (a particle range of one
// bunch).  The bunch's deferred 2.5D kick comes first (its op is assembled from the
// bunch's record and the batch's common factors), then the map program; extrema are
// reduced per work item.  Dynamic LDS: kBatchPhiLds doubles when the kick is active.
template <bool EXTREMA, int LEVEL>
__device__ __forceinline__ void push_batch_body(const BatchBunch* __restrict__ bb,
                                                const BatchItem* __restrict__ items,
                                                const ProgramWords<kProgWords>& prog,
                                                const BatchKick& kick,
                                                double* __restrict__ partials) {
  const BatchItem it = items[blockIdx.x];
  const BatchBunch& B = bb[it.bunch];
  // the kick's values for this step, before any store of the kernel (scalar loads)
  SC2DKickParams kp;
  if (kick.active) kp = sc2d_kick_params(B.st);
  const int nx = B.nx, ny = B.ny, nz = B.nz;
  const gptr<const double> gphi = to_global((const double*)B.phi);
  const gptr<const double> zg = to_global((const double*)B.zg);
  const gptr<const double> zd = to_global((const double*)B.zd);
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
  double hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  const gptr<double> cx = to_global(B.v.c[0]);
  const gptr<double> cxp = to_global(B.v.c[1]);
  const gptr<double> cy = to_global(B.v.c[2]);
  const gptr<double> cyp = to_global(B.v.c[3]);
  const gptr<double> cz = to_global(B.v.c[4]);
  const gptr<double> cdE = to_global(B.v.c[5]);
  extern __shared__ double sphi[];
  const bool lds_phi = kick.active && nx * ny <= kBatchPhiLds;
  if (lds_phi) {  // one load per thread and node slot, all in flight together
    constexpr int KP = kBatchPhiLds / kPushThreads;
    const int ng = nx * ny;
    double v[KP];
#pragma unroll
    for (int u = 0; u < KP; u++) {
      const int k = (int)threadIdx.x + u * kPushThreads;
      v[u] = gphi[k < ng ? k : 0];
    }
#pragma unroll
    for (int u = 0; u < KP; u++) {
      const int k = (int)threadIdx.x + u * kPushThreads;
      if (k < ng) sphi[k] = v[u];
    }
    __syncthreads();
  }
  int64_t i = it.begin + threadIdx.x;
  double q[6];
  if (i < it.end) load6(cx, cxp, cy, cyp, cz, cdE, i, q);
  for (; i < it.end; i += kPushThreads) {
    double x = q[0], xp = q[1], y = q[2], yp = q[3], z = q[4], dE = q[5];
    // this particle's kick loads, then the next particle's coordinates, then the arithmetic
    SC2DKickLoads L;
    if (lds_phi)
      sc2p5drb_kick_loads(kp, sphi, nx, ny, zg, zd, nz, x, y, z, L);
    else if (kick.active)
      sc2p5drb_kick_loads(kp, gphi, nx, ny, zg, zd, nz, x, y, z, L);
    if (i + kPushThreads < it.end) load6(cx, cxp, cy, cyp, cz, cdE, i + kPushThreads, q);
    if (kick.active) sc2p5drb_kick_apply(kp, L, nz, kick.p4, kick.p5, x, xp, y, yp, dE);
    run_program<LEVEL>(prog, x, xp, y, yp, z, dE);
    cx[i] = x;
    cxp[i] = xp;
    cy[i] = y;
    cyp[i] = yp;
    cz[i] = z;
    cdE[i] = dE;
    if (EXTREMA) {
      lo[0] = fmin(lo[0], x);
      hi[0] = fmax(hi[0], x);
      lo[1] = fmin(lo[1], y);
      hi[1] = fmax(hi[1], y);
      lo[2] = fmin(lo[2], z);
      hi[2] = fmax(hi[2], z);
    }
  }
  if (EXTREMA) block_extrema(lo, hi, partials);
}


// Levels 0 and 1 are bounded to three waves per SIMD (168 VGPRs): they take 121 to 141 without
// spills.  (With the interpreter of fixed op records they took 169, and the bound was 7%
// faster.)  Level 2 spilled 220 bytes at the bound then and was left out of it; by itself it
// now takes 157, with extrema 169, one register more than three waves allow.
template <bool EXTREMA, int LEVEL>
__global__ __launch_bounds__(kPushThreads) __attribute__((amdgpu_waves_per_eu(3))) void
push_batch_kernel(const BatchBunch* __restrict__ bb, const BatchItem* __restrict__ items,
                  ProgramWords<kProgWords> prog, BatchKick kick, double* __restrict__ partials) {
  push_batch_body<EXTREMA, LEVEL>(bb, items, prog, kick, partials);
}
template <bool EXTREMA>
__global__ __launch_bounds__(kPushThreads) void push_batch_kernel_l2(
    const BatchBunch* __restrict__ bb, const BatchItem* __restrict__ items,
    ProgramWords<kProgWords> prog, BatchKick kick, double* __restrict__ partials) {
  push_batch_body<EXTREMA, 2>(bb, items, prog, kick, partials);
}

}  // namespace

void launch_push_batch(const BatchBunch* bb, const BatchItem* items, int nitems,
                       const OpProgram& prog, const BatchKick& kick, double* partials,
                       int threads, hipStream_t s) {
  OB_REQUIRE(threads == kPushThreads, "batch push: unsupported block size");
  if (nitems == 0) return;
  const int level = prog.level;
  OB_REQUIRE(level <= 2, "batch push: a space-charge kick inside a map program");
  const size_t lds = kick.active ? sizeof(double) * kBatchPhiLds : 0;
  auto go = [&](auto kernel, double* part) {
    hipLaunchKernelGGL(kernel, dim3(nitems), dim3(kPushThreads), lds, s, bb, items,
                       static_cast<const ProgramWords<kProgWords>&>(prog), kick, part);
  };
  if (prog.want_extrema) {
    OB_REQUIRE(partials != nullptr, "batch push: extrema requested without a buffer");
    ProfScope ps("push_batch_extrema");
    if (level == 2)
      go(push_batch_kernel_l2<true>, partials);
    else if (level == 1)
      go(push_batch_kernel<true, 1>, partials);
    else
      go(push_batch_kernel<true, 0>, partials);
  } else {
    if (prog.words == 0 && !kick.active) return;
    ProfScope ps("push_batch");
    if (level == 2)
      go(push_batch_kernel_l2<false>, nullptr);
    else if (level == 1)
      go(push_batch_kernel<false, 1>, nullptr);
    else
      go(push_batch_kernel<false, 0>, nullptr);
  }
  OB_HIP(hipGetLastError());
}

int push_grid_blocks(int64_t n) {
  int64_t b = (n + kPushThreads - 1) / kPushThreads;
  if (b < 1) b = 1;
  if (b > kMaxPushBlocks) b = kMaxPushBlocks;
  return (int)b;
}

int launch_push(const DeviceBunchView& v, const OpProgram& prog, const Op* kick0,
                double* ext_partials, hipStream_t s) {
  // With a leading 2.5D kick, four waves per SIMD fit and 1024 workgroups are resident at once:
  // more only wait, each with the latency of its first loads and a row of extrema for the
  // next kernel to read (1M particles, 200 x 150 nodes: push 34.5 us with 3907 workgroups, 31.7
  // with 1024, 33.8 with 512; the deposit that reads the rows 26.9, 25.7, 25.6).  Maps alone
  // fit more waves: a ring's programs take 208 us with 3907 workgroups, 244 with 1024.
  const int blocks = std::min(push_grid_blocks(v.n), kick0 ? kKickPushBlocks : kMaxPushBlocks);
  const bool ext = prog.want_extrema != 0;
  OB_REQUIRE(!ext || ext_partials != nullptr, "push: extrema requested without a buffer");
  if (!ext && ((prog.words == 0 && !kick0) || v.n == 0)) return 0;
  Kick0 k{};
  if (kick0)
    k = Kick0{op_ptr<const SC2DState*>(kick0->p[0]), op_ptr<const double*>(kick0->p[1]),
              op_ptr<const double*>(kick0->p[2]), op_ptr<const double*>(kick0->p[3]),
              kick0->p[4], kick0->p[5], kick0->i0, kick0->i1, kick0->i2, 0};
  ProgramWords<kProgSmallWords> small;
  const bool fits = prog.words <= kProgSmallWords;
  if (fits) std::memcpy(&small, &prog, offsetof(ProgramWords<kProgSmallWords>, data) +
                                           sizeof(double) * prog.words);
  ProfScope ps(ext ? "push_extrema" : "push");
  auto go = [&](auto ce, auto cl, auto ck) {
    constexpr bool E = decltype(ce)::value != 0, K = decltype(ck)::value != 0;
    constexpr int L = decltype(cl)::value;
    if (fits)
      hipLaunchKernelGGL((push_kernel<E, L, K, kProgSmallWords>), dim3(blocks),
                         dim3(kPushThreads), 0, s, v, small, k, ext_partials);
    else
      hipLaunchKernelGGL((push_kernel<E, L, K, kProgWords>), dim3(blocks), dim3(kPushThreads), 0,
                         s, v, static_cast<const ProgramWords<kProgWords>&>(prog), k,
                         ext_partials);
  };
  auto by_level = [&](auto ce, auto ck) {
    if (prog.level == 0)
      go(ce, std::integral_constant<int, 0>{}, ck);
    else if (prog.level == 1)
      go(ce, std::integral_constant<int, 1>{}, ck);
    else if (prog.level == 2)
      go(ce, std::integral_constant<int, 2>{}, ck);
    else
      go(ce, std::integral_constant<int, 3>{}, ck);
  };
  using No = std::integral_constant<int, 0>;
  using Yes = std::integral_constant<int, 1>;
  if (ext)
    kick0 ? by_level(Yes{}, Yes{}) : by_level(Yes{}, No{});
  else
    kick0 ? by_level(No{}, Yes{}) : by_level(No{}, No{});
  OB_HIP(hipGetLastError());
  return blocks;
}

int launch_tile_push(const DeviceBunchView& v, const TileKick& t, const OpProgram& prog,
                     double* ext_partials, hipStream_t s) {
  OB_REQUIRE(v.n == t.n, "tile kick: the bunch has changed since its sort");
  OB_REQUIRE(prog.level <= 1 && prog.words <= kProgSmallWords, "tile kick: program too long");
  const bool ext = prog.want_extrema != 0;
  OB_REQUIRE(!ext || ext_partials != nullptr, "push: extrema requested without a buffer");
  const size_t lds = tile_lds_bytes(t.g);
  const int blocks = (int)std::min<int64_t>(t.max_items + 1, kMaxPushBlocks);
  ProgramWords<kProgSmallWords> small;
  std::memcpy(&small, &prog, offsetof(ProgramWords<kProgSmallWords>, data) +
                                 sizeof(double) * prog.words);
  ProfScope ps(prog.words || ext ? (ext ? "tile_push_extrema" : "tile_push") : "tile_kick");
  auto go = [&](auto cb, auto ce, auto cl, auto cm) {
    constexpr bool B = decltype(cb)::value != 0, E = decltype(ce)::value != 0;
    constexpr bool M = decltype(cm)::value != 0;
    constexpr int L = decltype(cl)::value;
    static bool ready = false;
    if (!ready) {  // (extrema: 192 static bytes beside the block of phi)
      OB_HIP(hipFuncSetAttribute((const void*)tile_push<B, E, L, M>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024));
      ready = true;
    }
    hipLaunchKernelGGL((tile_push<B, E, L, M>), dim3(blocks), dim3(kTileThreads), lds, s, v.c[0],
                       (int64_t)(v.c[1] - v.c[0]), t, small, ext_partials);
  };
  using No = std::integral_constant<int, 0>;
  using Yes = std::integral_constant<int, 1>;
  auto by_bnd = [&](auto... r) { t.k.bnd_type ? go(Yes{}, r...) : go(No{}, r...); };
  if (!ext && prog.words == 0)
    by_bnd(No{}, No{}, No{});
  else if (prog.level == 1)
    ext ? by_bnd(Yes{}, Yes{}, Yes{}) : by_bnd(No{}, Yes{}, Yes{});
  else
    ext ? by_bnd(Yes{}, No{}, Yes{}) : by_bnd(No{}, No{}, Yes{});
  OB_HIP(hipGetLastError());
  return blocks;
}

namespace {
double word_of(uint32_t lo, uint32_t hi) {
  const uint64_t u = (uint64_t)lo | ((uint64_t)hi << 32);
  double d;
  std::memcpy(&d, &u, sizeof(d));
  return d;
}
// What an op takes from the program and does to it: the coefficients dpc and g2i it was queued
// with (0: none), whether it reads dp/p or 1/(1 + dp/p), whether it changes dE.
struct OpUse {
  double dpc = 0.0, g2i = 0.0;
  bool has_dpc = false, has_g2i = false, reads = false, moves_dE = false;
};
}  // namespace

size_t program_encode(const Op* ops, size_t count, OpProgram& prog) {
  prog.words = 0;
  prog.want_extrema = 0;
  prog.level = 0;
  prog.dpc = prog.g2i = 0.0;
  double cur_dpc = 0.0, cur_g2i = 0.0;
  bool has_dpc = false, has_g2i = false, env_used = false, fresh = false;
  auto same = [](double a, double b) { return std::memcmp(&a, &b, sizeof(a)) == 0; };
  int n = 0;
  size_t k = 0;
  for (; k < count; k++) {
    const Op& o = ops[k];
    OpUse u;
    double q[16];
    int nq = 0;
    uint32_t ia = 0;
    auto put = [&](double v) { q[nq++] = v; };
    auto dpc = [&](double v) { u.dpc = v; u.has_dpc = true; u.reads = true; };
    auto g2i = [&](double v) { u.g2i = v; u.has_g2i = true; };
    switch (o.kind) {
      case OP_DRIFT: put(o.p[0]); g2i(o.p[1]); dpc(o.p[2]); break;
      case OP_QUAD1:  // m11 = m22 and m33 = m44 are one value each
        for (int j : {0, 1, 2, 4, 5, 6, 9}) put(o.p[j]);
        g2i(o.p[8]);
        dpc(o.p[10]);
        break;
      case OP_QUAD2: put(o.p[0]); g2i(o.p[1]); dpc(o.p[2]); break;
      case OP_QUADFRINGE_IN:
      case OP_QUADFRINGE_OUT: put(o.p[1]); dpc(o.p[0]); break;
      case OP_MULTP:
        put(o.p[0]);
        ia = (uint32_t)o.i0 | (o.i1 ? 256u : 0u);
        break;
      case OP_MULTPFRINGE_IN:
      case OP_MULTPFRINGE_OUT:
        put(o.p[1]); put(o.p[2]); dpc(o.p[0]);
        ia = (uint32_t)o.i0;
        break;
      case OP_WRAPBUNCH: put(o.p[0]); break;
      case OP_ROTATEXY: put(o.p[0]); put(o.p[1]); break;
      case OP_KICK:
        for (int j = 0; j < 3; j++) put(o.p[j]);
        u.moves_dE = o.p[2] != 0.;
        break;
      case OP_SC2P5DRB_KICK:
        for (int j = 0; j < 6; j++) put(o.p[j]);
        put(word_of((uint32_t)o.i1, (uint32_t)o.i2));
        ia = (uint32_t)o.i0;
        u.moves_dE = true;
        break;
      case OP_SC3D_KICK:
        for (int j = 0; j < 12; j++) put(o.p[j]);
        put(word_of((uint32_t)o.i1, (uint32_t)o.i2));
        ia = (uint32_t)o.i0;
        u.moves_dE = true;
        break;
      case OP_BEND1:
        for (int j = 0; j < 10; j++) put(o.p[j]);
        dpc(o.p[10]);
        break;
      case OP_BEND3: put(o.p[0]); g2i(o.p[1]); dpc(o.p[2]); break;
      case OP_BEND4: put(o.p[0]); dpc(o.p[1]); break;
      case OP_BENDFRINGE_IN:
      case OP_BENDFRINGE_OUT: put(o.p[0]); dpc(o.p[1]); break;
      case OP_WEDGEROTATE:
        put(o.p[0]); put(o.p[1]);
        u.dpc = o.p[2];
        u.has_dpc = true;
        ia = (uint32_t)o.i0;
        u.moves_dE = true;
        break;
      case OP_WEDGEDRIFT:
        put(o.p[0]); dpc(o.p[1]); g2i(o.p[2]);
        ia = (uint32_t)o.i0;
        break;
      case OP_WEDGEBEND: {
        const int nm = (o.i0 >> 1) & 15;
        put(o.p[0]); put(o.p[1]);
        put(word_of((uint32_t)o.i2, (uint32_t)o.i1));
        for (int l = 0; l < nm; l++) put(o.p[4 + l]);
        dpc(o.p[2]); g2i(o.p[3]);
        ia = (uint32_t)o.i0;
        break;
      }
      case OP_SOLN: put(o.p[0]); put(o.p[1]); g2i(o.p[2]); dpc(o.p[3]); break;
      case OP_RINGRF:
        for (int j = 0; j < 5; j++) put(o.p[j]);
        u.moves_dE = true;
        break;
      default: throw Error{"map program: unknown op"};
    }
    // the program's coefficients are the first ones; others are set by an OP_ENV before the op
    const bool env = (u.has_dpc && (has_dpc || env_used) && !same(u.dpc, cur_dpc)) ||
                     (u.has_g2i && (has_g2i || env_used) && !same(u.g2i, cur_g2i));
    if (n + (env ? 3 : 0) + 1 + nq > kProgWords) break;
    if (env) {
      if (u.has_dpc && !same(u.dpc, cur_dpc)) fresh = false;
      if (u.has_dpc) cur_dpc = u.dpc;
      if (u.has_g2i) cur_g2i = u.g2i;
      prog.data[n++] = word_of((uint32_t)OP_ENV | (3u << 12), 0u);
      prog.data[n++] = cur_dpc;
      prog.data[n++] = cur_g2i;
      env_used = true;
    } else if (!env_used) {
      if (u.has_dpc) prog.dpc = cur_dpc = u.dpc;
      if (u.has_g2i) prog.g2i = cur_g2i = u.g2i;
    }
    has_dpc = has_dpc || u.has_dpc;
    has_g2i = has_g2i || u.has_g2i;
    uint32_t h = (uint32_t)o.kind | ((uint32_t)(1 + nq) << 12);
    if (u.reads && !fresh) {
      h |= kProgRecalc;
      fresh = true;
    }
    if (u.moves_dE) fresh = false;
    prog.data[n++] = word_of(h, ia);
    for (int j = 0; j < nq; j++) prog.data[n++] = q[j];
    prog.level = std::max(prog.level, op_level(o.kind));
  }
  prog.words = n;
  return k;
}

}  // namespace ob
