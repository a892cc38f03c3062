// ob_diag.hip -- bunch diagnostics on the device: the moments of BunchTwissAnalysis
// (src/orbit/BunchDiagnostics/BunchTwissAnalysis.cc:49-142), its x-y power moments
// (computeBunchMoments, :145-337), the six coordinate extrema of BunchExtremaCalculator
// (src/utils/bunch/BunchExtremaCalculator.cc:37-120) and Grid1D::binBunch along any axis
// (src/spacecharge/Grid1D.cc:241-275, 328-352), which the profile diagnostics use.
//
// analyzeBunch sums, over the particles, the weight (macrosize attribute or 1), the
// weighted coordinates and the weighted products of coordinate pairs.  Here each
// workgroup sums its particles in registers and writes its 28 partial sums; one workgroup
// adds the partials in a fixed order.  The host derives averages, correlations and
// emittances exactly as the reference does, without downloading the 6 x N coordinates.
#include <algorithm>
#include <cmath>

#include "ob_internal.hpp"
#include "ob_sc_device.hpp"

namespace ob {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxBlocks = 1024;
constexpr int kSums = 28;  // weight, 6 first moments, 21 products (i <= j)

// Sums of NV values over the workgroup's kThreads threads: each wave adds its lanes with
// shuffles (the NV chains are independent, so their latencies overlap), one barrier, then
// thread k < NV adds the waves' sums of value k in wave order and stores it to out[k].  A
// barrier pair per value instead made the 28 sums cost as much as reading the particles.
template <int NV>
__device__ __forceinline__ void block_sums(double (&s)[NV], double* sh, double* __restrict__ out) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < NV; k++) s[k] += __shfl_xor(s[k], o, 64);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) sh[w * NV + k] = s[k];
  __syncthreads();
  if (threadIdx.x < NV) {
    double t = 0.0;
    for (int j = 0; j < kThreads / 64; j++) t += sh[j * NV + threadIdx.x];
    out[threadIdx.x] = t;
  }
}

// Two particles per thread and round: twice the loads in flight (a masked lane reloads the
// first particle with weight 0, and NaN or infinite coordinates of it are not touched).
__global__ __launch_bounds__(kThreads) void moment_partials(DeviceBunchView v,
                                                            double* __restrict__ part) {
  __shared__ double sh[kThreads / 64 * kSums];
  double s[kSums];
#pragma unroll
  for (int k = 0; k < kSums; k++) s[k] = 0.0;
  gptr<const double> c[6];
#pragma unroll
  for (int k = 0; k < 6; k++) c[k] = to_global((const double*)v.c[k]);
  const gptr<const double> pm = to_global((const double*)v.msize);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  constexpr int U = 2;
  for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < v.n; i0 += U * stride) {
    double q[U][6], w[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = i0 + u * stride < v.n ? i0 + u * stride : i0;
#pragma unroll
      for (int k = 0; k < 6; k++) q[u][k] = c[k][i];
      w[u] = pm ? pm[i] : 1.0;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (i0 + u * stride >= v.n) break;
      s[0] += w[u];
#pragma unroll
      for (int k = 0; k < 6; k++) s[1 + k] += w[u] * q[u][k];
      int p = 7;
#pragma unroll
      for (int a = 0; a < 6; a++)
#pragma unroll
        for (int b = a; b < 6; b++) s[p++] += w[u] * q[u][a] * q[u][b];
    }
  }
  block_sums<kSums>(s, sh, part + (size_t)blockIdx.x * kSums);
}

// Rows part[nblk][nt] added (OP 0) or their extrema taken (OP 1: min of even columns, max
// of odd ones; OP 2: max) per column, nt <= 128.  One workgroup: kRedThreads / C threads
// per column (C = nt rounded up to a power of two) walk the rows, eight loads in flight,
// and meet in LDS in row-group order, so the result does not depend on timing.  The former
// form, one thread per column walking up to 1024 rows one load at a time, took 215-235 us
// for any bunch of 262k particles or more; this one takes 8-9 us.  seq_out, if given: a
// host word that gets seq once the result is written (pinned memory).
constexpr int kRedThreads = 1024;
template <int OP>
__device__ __forceinline__ double red_op(double a, double b, int k) {
  if (OP == 0) return a + b;
  if (OP == 1 && !(k & 1)) return b < a ? b : a;
  return b > a ? b : a;
}
template <int OP>
__device__ __forceinline__ double red_init(int k) {
  return OP == 0 ? 0.0 : (OP == 2 ? 0.0 : ((k & 1) ? -DBL_MAX : DBL_MAX));
}
template <int OP>
__global__ __launch_bounds__(kRedThreads) void row_reduce(const double* __restrict__ part,
                                                          int nblk, int nt, int cbits,
                                                          double* __restrict__ out,
                                                          uint64_t* __restrict__ seq_out,
                                                          uint64_t seq) {
  __shared__ double sh[kRedThreads];
  const int C = 1 << cbits, k = threadIdx.x & (C - 1), r = threadIdx.x >> cbits;
  const int g = kRedThreads >> cbits;
  double acc = red_init<OP>(k);
  if (k < nt) {
    int b = r;
    for (; b + 7 * g < nblk; b += 8 * g) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = part[(size_t)(b + u * g) * nt + k];
#pragma unroll
      for (int u = 0; u < 8; u++) acc = red_op<OP>(acc, v[u], k);
    }
    for (; b < nblk; b += g) acc = red_op<OP>(acc, part[(size_t)b * nt + k], k);
  }
  sh[threadIdx.x] = acc;
  for (int h = g >> 1; h > 0; h >>= 1) {
    __syncthreads();
    if (r < h) sh[threadIdx.x] = red_op<OP>(sh[threadIdx.x], sh[threadIdx.x + (h << cbits)], k);
  }
  if (r == 0 && k < nt) out[k] = sh[k];
  if (seq_out) {  // the total is visible to the host before the number it watches
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(seq_out, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ---- extrema of the six coordinates -------------------------------------------------
// Per workgroup: min and max of x, xp, y, yp, z, dE (12 values, min/max interleaved);
// comparisons as in the reference (a value replaces the extremum only if strictly beyond).
__device__ __forceinline__ double lo(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double hi(double a, double b) { return b > a ? b : a; }

__global__ __launch_bounds__(kThreads) void extrema6_partials(DeviceBunchView v,
                                                              double* __restrict__ part) {
  __shared__ double sh[kThreads / 64][12];
  double e[12];
  gptr<const double> c[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    e[2 * k] = DBL_MAX;
    e[2 * k + 1] = -DBL_MAX;
    c[k] = to_global((const double*)v.c[k]);
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  constexpr int U = 2;  // a masked lane reloads the first particle: it cannot change an extremum
  for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < v.n; i0 += U * stride) {
    double q[U][6];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = i0 + u * stride < v.n ? i0 + u * stride : i0;
#pragma unroll
      for (int k = 0; k < 6; k++) q[u][k] = c[k][i];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int k = 0; k < 6; k++) {
        e[2 * k] = lo(e[2 * k], q[u][k]);
        e[2 * k + 1] = hi(e[2 * k + 1], q[u][k]);
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 6; k++) {
      e[2 * k] = lo(e[2 * k], __shfl_xor(e[2 * k], o, 64));
      e[2 * k + 1] = hi(e[2 * k + 1], __shfl_xor(e[2 * k + 1], o, 64));
    }
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 12; k++) sh[threadIdx.x >> 6][k] = e[k];
  __syncthreads();
  if (threadIdx.x < 12) {
    const int k = threadIdx.x;
    double r = sh[0][k];
    for (int w = 1; w < kThreads / 64; w++) r = (k & 1) ? hi(r, sh[w][k]) : lo(r, sh[w][k]);
    part[(size_t)blockIdx.x * 12 + k] = r;
  }
}

// ---- extremaR: largest distance from the mean transverse position -----------------------
// Per-workgroup sums of x and y (unweighted, as the reference's mean), their total
// (row_reduce), each workgroup's largest distance from the mean, the largest of those.
__global__ __launch_bounds__(kThreads) void xy_sum_partials(DeviceBunchView v,
                                                            double* __restrict__ part) {
  __shared__ double sh[kThreads / 64 * 2];
  double s[2] = {0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < v.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    s[0] += v.c[0][i];
    s[1] += v.c[2][i];
  }
  block_sums<2>(s, sh, part + 2 * (size_t)blockIdx.x);
}

__global__ __launch_bounds__(kThreads) void rmax_partials(DeviceBunchView v,
                                                          const double* __restrict__ sums,
                                                          double* __restrict__ part) {
  __shared__ double sh[kThreads / 64];
  const double xa = sums[0] / (double)v.n, ya = sums[1] / (double)v.n;
  double r = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < v.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double dx = v.c[0][i] - xa, dy = v.c[2][i] - ya;
    const double ri = sqrt(dx * dx + dy * dy);
    r = ri > r ? ri : r;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_xor(r, o, 64);
    r = t > r ? t : r;
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; w++) r = sh[w] > r ? sh[w] : r;
    part[blockIdx.x] = r;
  }
}

// ---- Grid1D::binBunch along one coordinate --------------------------------------------
// Linear (cloud-in-cell) weights of Grid1D::binValue (Grid1D.cc:422-440) with the grid's
// periodic wrap at both ends.  Grids up to kBinLds bins accumulate a private histogram per
// workgroup in LDS and write it out; a second pass adds the workgroups' histograms bin by
// bin in a fixed order.  Larger grids add into one global histogram with atomics.
constexpr int kBinLds = 4096;  // 32 KiB of FP64 bins per workgroup

struct Bin1D {
  int axis, by_particle, nz;
  double value;  // bunch macrosize when the bunch has no macrosize attribute
  double zMin, zMax, dz;
};

template <bool LDS>
__global__ __launch_bounds__(kThreads) void bin1d_partials(DeviceBunchView v, Bin1D g,
                                                           double* __restrict__ part) {
  extern __shared__ double hist[];
  double* h = LDS ? hist : part;
  if (LDS) {
    for (int k = threadIdx.x; k < g.nz; k += blockDim.x) hist[k] = 0.0;
    __syncthreads();
  }
  const double* __restrict__ zc = v.c[g.axis];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < v.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double z = zc[i];
    if (z < g.zMin || z > g.zMax) continue;
    const double val = g.by_particle ? 1.0 : (v.msize ? v.msize[i] : g.value);
    int i0, ip;
    double w0, wp;
    grid1d_ind_wz(z, g.zMin, g.dz, g.nz, i0, ip, w0, wp);
    if (g.nz > 1) {
      atomicAdd(&h[i0], w0 * val);
      atomicAdd(&h[ip], wp * val);
    } else {
      atomicAdd(&h[i0], val);
    }
  }
  if (LDS) {
    __syncthreads();
    for (int k = threadIdx.x; k < g.nz; k += blockDim.x)
      part[(size_t)blockIdx.x * g.nz + k] = hist[k];
  }
}

// Sixteen bins per workgroup (128-byte row segments), sixteen row groups per bin with eight
// loads in flight each, added in row-group order: 115 us as one thread per bin walking 512
// rows (128 bins: half a workgroup on the whole chip), 4 us so.
constexpr int kBinCols = 16;
__global__ __launch_bounds__(kThreads) void bin1d_reduce(const double* __restrict__ part,
                                                         int nblk, int nz,
                                                         double* __restrict__ out) {
  __shared__ double sh[kThreads];
  constexpr int g = kThreads / kBinCols;
  const int k = blockIdx.x * kBinCols + (int)threadIdx.x % kBinCols;
  const int r = (int)threadIdx.x / kBinCols;
  double s = 0.0;
  if (k < nz) {
    int b = r;
    for (; b + 7 * g < nblk; b += 8 * g) {
      double t[8];
#pragma unroll
      for (int u = 0; u < 8; u++) t[u] = part[(size_t)(b + u * g) * nz + k];
#pragma unroll
      for (int u = 0; u < 8; u++) s += t[u];
    }
    for (; b < nblk; b += g) s += part[(size_t)b * nz + k];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (r == 0 && k < nz) {
    for (int j = 1; j < g; j++) s += sh[j * kBinCols + threadIdx.x];
    out[k] = s;
  }
}

// ---- computeBunchMoments: sums of x-y power products --------------------------------
// BunchTwissAnalysis::computeBunchMoments (BunchTwissAnalysis.cc:145-337) accumulates, for
// j < order and i <= order - j, momX[i] / xb^i * momY[j] / yb^j over the particles, with
// momX[i] = prod (m (x - D dE / (E + M) / beta^2 - <x>)) and momY[j] = prod (m (y - <y>))
// (m = 1 without the macrosize attribute); with the attribute each term also adds
// momX[i] momY[j].  Without the attribute the statement after the loops adds
// momX[2] momY[order] to entry [2][order] once per particle (it sits outside the braces).
// The kernel adds momX[i] momY[j] (the divisors are the same for every particle: the host
// divides the sums once, two roundings instead of three per particle), each thread's sums
// in registers for the order it is compiled for.  Sums in LDS columns with two divisions
// per term and particle took 57 us at 1M particles and order 4, against 16 us.
constexpr int kMaxMomOrder = 12;
__host__ __device__ constexpr int mom_terms(int order) { return order * (order + 3) / 2; }

struct XYMom {
  int disp, stray;
  double xAvg, yAvg, D, Em, b2;  // Em = E_kin + mass, b2 = beta^2
};

template <int ORDER>
__global__ __launch_bounds__(kThreads) void xy_moment_partials(DeviceBunchView v, XYMom p,
                                                               double* __restrict__ part) {
  constexpr int NT = mom_terms(ORDER) + 2;
  __shared__ double sh[kThreads / 64 * NT];
  double s[NT];
#pragma unroll
  for (int k = 0; k < NT; k++) s[k] = 0.0;
  const gptr<const double> cx = to_global((const double*)v.c[0]);
  const gptr<const double> cy = to_global((const double*)v.c[2]);
  const gptr<const double> cd = to_global((const double*)v.c[5]);
  const gptr<const double> pm = to_global((const double*)v.msize);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < v.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double m = pm ? pm[i] : 1.0;
    const double dispterm = p.disp ? p.D * cd[i] / p.Em / p.b2 : 0.0;
    const double dx = (cx[i] - dispterm) - p.xAvg;
    const double dy = cy[i] - p.yAvg;
    const double fx = pm ? m * dx : dx, fy = pm ? m * dy : dy;
    double mX[ORDER + 1];
    mX[0] = 1.0;
#pragma unroll
    for (int a = 1; a <= ORDER; a++) mX[a] = mX[a - 1] * fx;
    double mY = 1.0;
    int k = 0;
#pragma unroll
    for (int j = 0; j < ORDER; j++) {
#pragma unroll
      for (int a = 0; a <= ORDER - j; a++) s[k++] += mX[a] * mY;
      mY = mY * fy;
    }
    if (p.stray) s[NT - 2] += dx * dx * mY;  // momX[2] momY[order]
    s[NT - 1] += m;
  }
  block_sums<NT>(s, sh, part + (size_t)blockIdx.x * NT);
}

// Scratch of ob_bunch_moments_noalloc: the per-workgroup partial sums (at most kMaxBlocks
// rows of kSums) and their total, 229,600 bytes whatever the bunch size.
constexpr size_t kScratchDoubles = (size_t)(kMaxBlocks + 1) * kSums;

}  // namespace
}  // namespace ob

// Held by every device the library runs on until the process ends.  In host code this name
// is a host-side stand-in, not a device address: host code uses the address looked up by
// diag_scratch_setup for the current device.
static __device__ __align__(256) double scratch[ob::kScratchDoubles];

namespace ob {
namespace {
constexpr int kMaxDevices = 64;
double* g_scratch_dev[kMaxDevices] = {};

// Column sums or extrema (row_reduce) of part[nblk][nt] into out[nt].
template <int OP>
void launch_row_reduce(const double* part, int nblk, int nt, double* out, hipStream_t s,
                       uint64_t* seq_out = nullptr, uint64_t seq = 0) {
  int cbits = 0;
  while ((1 << cbits) < nt) cbits++;
  OB_REQUIRE(cbits <= 7, "row_reduce: more than 128 columns");
  hipLaunchKernelGGL(row_reduce<OP>, dim3(1), dim3(kRedThreads), 0, s, part, nblk, nt, cbits, out,
                     seq_out, seq);
}

// The total of part[nblk][nt] to the host array out[nt] through the bunch's pinned words:
// no copy command and no wait for the stream to drain.
template <int OP>
void rows_to_host(DiagWork& w, const double* part, int nblk, int nt, double* out,
                  hipStream_t s) {
  const uint64_t want = ++w.seq;
  launch_row_reduce<OP>(part, nblk, nt, w.host_dev + 1, s,
                        reinterpret_cast<uint64_t*>(w.host_dev), want);
  OB_HIP(hipGetLastError());
  host_wait_seq(reinterpret_cast<uint64_t*>(w.host), want, s);
  std::memcpy(out, w.host + 1, sizeof(double) * nt);
}

// Partial sums into buf[0 .. nblk * kSums), their total at buf + nblk * kSums, copied to
// the host array out[kSums]; waits for the copy.  Every partial row and the total are
// written before they are read, so buf needs no clearing.  Not recorded in the kernel
// profiler (which creates HIP events when it is on).
void moments_into(const DeviceBunchView& v, int nblk, double* buf, double* out, hipStream_t s) {
  hipLaunchKernelGGL(moment_partials, dim3(nblk), dim3(kThreads), 0, s, v, buf);
  launch_row_reduce<0>(buf, nblk, kSums, buf + (size_t)nblk * kSums, s);
  OB_HIP(hipGetLastError());
  OB_HIP(hipMemcpyAsync(out, buf + (size_t)nblk * kSums, sizeof(double) * kSums,
                        hipMemcpyDeviceToHost, s));
  OB_HIP(hipStreamSynchronize(s));
}
}  // namespace

void diag_scratch_setup(int device) {
  OB_REQUIRE(device >= 0 && device < kMaxDevices, "device index out of range");
  if (g_scratch_dev[device] != nullptr) return;
  double* p = nullptr;
  OB_HIP(hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)));
  OB_REQUIRE(p != nullptr, "no device address for the moments scratch");
  g_scratch_dev[device] = p;
}
}  // namespace ob

#define OB_API extern "C" __attribute__((visibility("default")))
#define OB_TRY try {
#define OB_CATCH               \
  }                            \
  catch (const ob::Error& e) { \
    ob::set_error(e.msg);      \
    return 1;                  \
  }                            \
  return 0;

// out[0] = sum of weights, out[1..6] = sum w c_k, out[7..27] = sum w c_a c_b (a <= b,
// row by row), weight = macrosize attribute or 1 (BunchTwissAnalysis.cc:49-142).
OB_API int ob_bunch_moments(ob_bunch* b, double* out) {
  OB_TRY OB_REQUIRE(b != nullptr && out != nullptr, "null handle");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  hipStream_t s = ob::stream();
  if (v.n == 0) {
    for (int k = 0; k < ob::kSums; k++) out[k] = 0.0;
    return 0;
  }
  const int nblk =
      (int)std::min<int64_t>(ob::kMaxBlocks, (v.n + ob::kThreads - 1) / ob::kThreads);
  ob::DiagWork& w = ob::bunch_diag_work(b, (size_t)nblk * ob::kSums);
  {
    ob::ProfScope ps("moment_partials");
    hipLaunchKernelGGL(ob::moment_partials, dim3(nblk), dim3(ob::kThreads), 0, s, v, w.dev);
  }
  ob::rows_to_host<0>(w, w.dev, nblk, ob::kSums, out, s);
  OB_CATCH
}

// ob_bunch_moments without any allocation: the partial sums go to the library's fixed
// device scratch (229,600 bytes per device).  Calls that overlap on one device race on
// that scratch.  A batched bunch is refused (its flush may rebuild the batch's records).
OB_API int ob_bunch_moments_noalloc(ob_bunch* b, double* out) {
  OB_TRY OB_REQUIRE(b != nullptr && out != nullptr, "null handle");
  OB_REQUIRE(!ob::bunch_in_batch(b),
             "ob_bunch_moments_noalloc: the bunch belongs to a batch; use ob_bunch_moments");
  int dev = -1;
  OB_HIP(hipGetDevice(&dev));
  OB_REQUIRE(dev >= 0 && dev < ob::kMaxDevices && ob::g_scratch_dev[dev] != nullptr,
             "ob_bunch_moments_noalloc: the library is not initialised on this device");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  if (v.n == 0) {
    for (int k = 0; k < ob::kSums; k++) out[k] = 0.0;
    return 0;
  }
  const int nblk =
      (int)std::min<int64_t>(ob::kMaxBlocks, (v.n + ob::kThreads - 1) / ob::kThreads);
  const size_t need = (size_t)(nblk + 1) * ob::kSums;
  OB_REQUIRE(need <= ob::kScratchDoubles,
             "ob_bunch_moments_noalloc: " + std::to_string(need) +
                 " doubles of scratch needed, the maximum is " +
                 std::to_string(ob::kScratchDoubles));
  ob::moments_into(v, nblk, ob::g_scratch_dev[dev], out, ob::stream());
  OB_CATCH
}

// BunchExtremaCalculator::getExtremaXYZ and getExtremaXpYpdE (BunchExtremaCalculator.cc:37-120)
// in one pass: out[12] = min, max of x, xp, y, yp, z, dE; DBL_MAX, -DBL_MAX for an empty
// bunch, as in the reference.
OB_API int ob_bunch_extrema(ob_bunch* b, double* out) {
  OB_TRY OB_REQUIRE(b != nullptr && out != nullptr, "null handle");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  hipStream_t s = ob::stream();
  if (v.n == 0) {
    for (int k = 0; k < 6; k++) {
      out[2 * k] = DBL_MAX;
      out[2 * k + 1] = -DBL_MAX;
    }
    return 0;
  }
  const int nblk =
      (int)std::min<int64_t>(ob::kMaxBlocks, (v.n + ob::kThreads - 1) / ob::kThreads);
  ob::DiagWork& w = ob::bunch_diag_work(b, (size_t)nblk * 12);
  {
    ob::ProfScope ps("extrema6_partials");
    hipLaunchKernelGGL(ob::extrema6_partials, dim3(nblk), dim3(ob::kThreads), 0, s, v, w.dev);
  }
  ob::rows_to_host<1>(w, w.dev, nblk, 12, out, s);
  OB_CATCH
}

// Grid1D::binBunch(bunch, axis) / binBunchByParticle(bunch, axis) (Grid1D.cc:241-275,
// 335-352) on a grid of nz cells over [zMin, zMax]: the binned values are ADDED to the
// host array arr[nz], as the reference adds into its grid.  by_particle = 1 gives each
// particle weight 1; otherwise its macrosize attribute or the bunch macrosize.
OB_API int ob_grid1d_bin_bunch(ob_bunch* b, int axis, int by_particle, int nz, double zMin,
                               double zMax, double* arr) {
  OB_TRY OB_REQUIRE(b != nullptr && arr != nullptr, "null handle");
  OB_REQUIRE(axis >= 0 && axis <= 5, "Grid1D::binBunch: the axis index should be between 0 and 5");
  OB_REQUIRE(nz >= 1 && nz <= (1 << 26),
             "Grid1D.binBunch: the number of bins should be between 1 and 2^26");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  if (v.n == 0) return 0;
  const ob::SyncInfo sy = ob::bunch_sync(b);
  hipStream_t s = ob::stream();
  ob::Bin1D g;
  g.axis = axis;
  g.by_particle = by_particle ? 1 : 0;
  g.nz = nz;
  g.value = sy.macrosize;
  g.zMin = zMin;
  g.zMax = zMax;
  g.dz = (zMax - zMin) / nz;  // Grid1D::setGridZ (Grid1D.cc:89-94)
  const bool lds = nz <= ob::kBinLds;
  const int64_t want = (v.n + ob::kThreads - 1) / ob::kThreads;
  const int nblk = (int)std::min<int64_t>(lds ? 512 : ob::kMaxBlocks, want);
  if (lds) {
    ob::DiagWork& w = ob::bunch_diag_work(b, (size_t)nblk * nz, nz);
    {
      ob::ProfScope ps("bin1d_partials");
      hipLaunchKernelGGL(ob::bin1d_partials<true>, dim3(nblk), dim3(ob::kThreads),
                         sizeof(double) * nz, s, v, g, w.dev);
    }
    hipLaunchKernelGGL(ob::bin1d_reduce, dim3((nz + ob::kBinCols - 1) / ob::kBinCols),
                       dim3(ob::kThreads), 0, s, w.dev, nblk, nz, w.host_dev + 1);
    OB_HIP(hipGetLastError());
    OB_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < nz; k++) arr[k] += w.host[1 + k];
    return 0;
  }
  double* buf = nullptr;  // a large grid's histogram is not kept
  OB_HIP(hipMalloc((void**)&buf, sizeof(double) * nz));
  std::vector<double> h((size_t)nz);
  try {
    OB_HIP(hipMemsetAsync(buf, 0, sizeof(double) * nz, s));
    {
      ob::ProfScope ps("bin1d_partials");
      hipLaunchKernelGGL(ob::bin1d_partials<false>, dim3(nblk), dim3(ob::kThreads), 0, s, v, g,
                         buf);
    }
    OB_HIP(hipGetLastError());
    OB_HIP(hipMemcpyAsync(h.data(), buf, sizeof(double) * nz, hipMemcpyDeviceToHost, s));
    OB_HIP(hipStreamSynchronize(s));
  } catch (...) {
    (void)hipFree(buf);
    throw;
  }
  OB_HIP(hipFree(buf));
  for (int k = 0; k < nz; k++) arr[k] += h[(size_t)k];
  OB_CATCH
}

// BunchTwissAnalysis::computeBunchMoments (BunchTwissAnalysis.cc:145-337), the particle
// sums.  prm[8] = xAvg, yAvg, D_x, E_kin + mass, beta^2, xb, yb, dispersion flag (> 0:
// subtract D_x dE / (E_kin + mass) / beta^2 from x); xb, yb are sqrt(beta) or
// sqrt(beta emittance) as the caller chose.  out[order (order + 3) / 2 + 2] = the sums
// for j = 0 .. order-1, i = 0 .. order-j (j outer), then the [2][order] entry of a bunch
// without the macrosize attribute (order >= 2; else 0), then the total weight.
OB_API int ob_bunch_xy_moments(ob_bunch* b, int order, const double* prm, double* out) {
  OB_TRY OB_REQUIRE(b != nullptr && prm != nullptr && out != nullptr, "null handle");
  OB_REQUIRE(order >= 1 && order <= ob::kMaxMomOrder,
             "computeBunchMoments: order must be between 1 and 12");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  hipStream_t s = ob::stream();
  ob::XYMom p;
  const bool ms = v.msize != nullptr;
  p.disp = prm[7] > 0 ? 1 : 0;
  p.stray = (!ms && order >= 2) ? 1 : 0;
  p.xAvg = prm[0]; p.yAvg = prm[1]; p.D = prm[2]; p.Em = prm[3]; p.b2 = prm[4];
  const int nt = ob::mom_terms(order) + 2;
  if (v.n == 0) {
    for (int k = 0; k < nt; k++) out[k] = 0.0;
    return 0;
  }
  const int nblk =
      (int)std::min<int64_t>(ob::kMaxBlocks, (v.n + ob::kThreads - 1) / ob::kThreads);
  ob::DiagWork& w = ob::bunch_diag_work(b, (size_t)nblk * nt);
  {
    ob::ProfScope ps("xy_moment_partials");
    switch (order) {
#define OB_CASE(o)                                                                            \
  case o:                                                                                     \
    hipLaunchKernelGGL(ob::xy_moment_partials<o>, dim3(nblk), dim3(ob::kThreads), 0, s, v, p, \
                       w.dev);                                                                \
    break;
      OB_CASE(1) OB_CASE(2) OB_CASE(3) OB_CASE(4) OB_CASE(5) OB_CASE(6)
      OB_CASE(7) OB_CASE(8) OB_CASE(9) OB_CASE(10) OB_CASE(11) OB_CASE(12)
#undef OB_CASE
      default: break;
    }
  }
  ob::rows_to_host<0>(w, w.dev, nblk, nt, out, s);
  int k = 0;
  for (int j = 0; j < order; j++)
    for (int a = 0; a <= order - j; a++, k++) {
      const double raw = out[k];
      out[k] = raw / pow(prm[5], (double)a) / pow(prm[6], (double)j);
      if (ms) out[k] += raw;
    }
  OB_CATCH
}

// BunchExtremaCalculator::getExtremaR (BunchExtremaCalculator.cc:167-208): the largest
// distance sqrt((x - <x>)^2 + (y - <y>)^2) from the unweighted mean position; 0 for an
// empty bunch.
OB_API int ob_bunch_extrema_r(ob_bunch* b, double* rmax) {
  OB_TRY OB_REQUIRE(b != nullptr && rmax != nullptr, "null handle");
  ob::bunch_flush(b, nullptr);
  const ob::DeviceBunchView v = ob::bunch_device_view(b);
  hipStream_t s = ob::stream();
  if (v.n == 0) {
    *rmax = 0.0;
    return 0;
  }
  const int nblk =
      (int)std::min<int64_t>(ob::kMaxBlocks, (v.n + ob::kThreads - 1) / ob::kThreads);
  ob::DiagWork& w = ob::bunch_diag_work(b, 3 * (size_t)nblk + 2);
  double *sums = w.dev, *total = w.dev + 2 * (size_t)nblk, *rpart = total + 2;
  {
    ob::ProfScope ps("rmax_partials");
    hipLaunchKernelGGL(ob::xy_sum_partials, dim3(nblk), dim3(ob::kThreads), 0, s, v, sums);
    ob::launch_row_reduce<0>(sums, nblk, 2, total, s);
    hipLaunchKernelGGL(ob::rmax_partials, dim3(nblk), dim3(ob::kThreads), 0, s, v, total, rpart);
  }
  ob::rows_to_host<2>(w, rpart, nblk, 1, rmax, s);
  OB_CATCH
}
