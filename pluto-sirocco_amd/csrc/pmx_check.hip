// Arithmetic checks: the short operations of the Cartesian faces, the plain
// cooling integrator and the line force beside the general ones, on the same
// operands.  They call the functions the kernels call, from a translation
// unit of their own, so that the kernels' inlining does not depend on them.
#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "pmx_wind_host.h"

namespace pmx {
namespace wind {
namespace {

// Copies of host arrays on the device, freed with it.
struct DeviceArrays {
  std::vector<void*> held;
  hipError_t err = hipSuccess;
  ~DeviceArrays() {
    for (void* p : held) (void)hipFree(p);
  }
  template <class T>
  T* make(const T* src, long long n) {
    T* p = nullptr;
    if (err == hipSuccess) err = hipMalloc(&p, sizeof(T) * n);
    if (err != hipSuccess) return nullptr;
    held.push_back(p);
    if (src) err = hipMemcpy(p, src, sizeof(T) * n, hipMemcpyHostToDevice);
    return p;
  }
  template <class T>
  void read(T* dst, const T* src, long long n) {
    if (err == hipSuccess) err = hipMemcpy(dst, src, sizeof(T) * n, hipMemcpyDeviceToHost);
  }
  int result() const {
    if (err == hipSuccess) return 0;
    set_error(hipGetErrorString(err));
    return -1;
  }
};

dim3 blocks(long long n) { return dim3((unsigned)std::min<long long>((n + 255) / 256, 4096)); }

// ---------------------------------------------------------------------
// quotients and roots
// ---------------------------------------------------------------------
__global__ void quotient_check_kernel(const double* __restrict__ x, const double* __restrict__ c,
                                      long long n, unsigned long long* bad) {
  unsigned long long mine[3] = {0, 0, 0};
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double a = x[i], b = c[i], r = a / b, s = fabs(a);
    mine[0] += quot(a, b, recip(b)) != r;
    mine[1] += div2(a, recip2(b, 1.0 / b)) != r;
    double y;
    mine[2] += s > 0.0 && sqrt_mod(s, y) != sqrt(s);
  }
  for (int q = 0; q < 3; q++)
    if (mine[q]) atomicAdd(bad + q, mine[q]);
}

// ---------------------------------------------------------------------
// force multiplier
// ---------------------------------------------------------------------
// out: [power, M] of the short form, [power, M] of the general one
__global__ void force_check_kernel(const double* __restrict__ num, const double* __restrict__ dvds,
                                   long long n, Const k, double* __restrict__ out) {
  const PowSeries C = pow_series();
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double d = dvds[i], y = recip(d);
    int e;
    const PowNum a = pow_num_fast(num[i], C);
    const DD D = log2_dd_fast(d, C, e);
    out[i] = force_power_fast(k, a, d, y, D, C);
    out[n + i] = force_mult_fast(k, a, d, y, D, C);
    const double g = d > 0.0 ? force_power_shared(k, pow_num(num[i]), d, log2_dd(d)) : 0.0;
    out[2 * n + i] = g;
    out[3 * n + i] = g > 4400. ? 4400. : g;
  }
}

// ---------------------------------------------------------------------
// plain cooling integrator
// ---------------------------------------------------------------------
struct CoolCheck {
  const double *rho, *p, *xi, *dt, *pre;   // pre: [5][n] or null
  double *rate, *e, *p_out;                // Radiat(E0); [short, general]; [general, as taken]
  long long* calls;                        // [short, general, as taken]
  int* flags;
};

PMX_HD void check_cell(const Const& k, double t_x, const CoolCheck& c, long long n, long long i) {
  RadCell R;
  R.rho = c.rho[i];
  R.trc = 1.0;
  R.x1 = 1.0;
  R.xi_s = c.xi[i];
  R.tr_s = t_x;
  R.t = 5.0;      // Radiat takes xi and T_r from the cell
  for (int q = 0; q < 5; q++) R.pre[q] = c.pre ? c.pre[q * n + i] : 1.0;
  R.nev = 0;
  rad_prepare(k, R);
  const double p = c.p[i], dt = c.dt[i];
  double E0 = p / (k.gamma - 1.0), cand;
  const double k1 = radiat(k, R, E0);
  c.rate[i] = k1;
  int f = 0, bad = 0;
  c.e[i] = 0.0;
  c.calls[i] = 0;
  if (short_form(R, E0, dt)) {
    bool over = false;
    c.e[i] = integrate_cell<true>(k, R, dt, E0, k1, bad, over);
    c.calls[i] = R.nev;
    f = PMX_COOL_SHORT | (over ? PMX_COOL_OVER : 0) | (bad ? PMX_COOL_BAD_SHORT : 0);
  }
  R.nev = 1;
  bad = 0;
  bool over = false;
  const double E1 = integrate_cell<false>(k, R, dt, E0, k1, bad, over);
  c.e[n + i] = E1;
  c.calls[n + i] = R.nev;
  f |= bad ? PMX_COOL_BAD_GENERAL : 0;
  c.p_out[i] = finish_cell(k, R, p, E1, dt, cand);
  R.nev = 0;
  bad = 0;
  c.p_out[n + i] = plain_cell(k, R, p, dt, cand, bad);
  c.calls[2 * n + i] = R.nev;
  c.flags[i] = f | (bad ? PMX_COOL_BAD_TAKEN : 0);
}

__global__ __launch_bounds__(128) void cool_check_kernel(Const k, double t_x, CoolCheck c,
                                                         long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) check_cell(k, t_x, c, n, i);
}

}  // namespace
}  // namespace wind
}  // namespace pmx

using namespace pmx;
using namespace pmx::wind;

extern "C" {

int pmx_check_quotients(const double* x, const double* c, long long n, long long* mismatches) {
  if (!x || !c || n <= 0 || !mismatches) { set_error("bad argument"); return -1; }
  DeviceArrays d;
  unsigned long long bad[3] = {0, 0, 0};
  const double *dx = d.make(x, n), *dc = d.make(c, n);
  unsigned long long* db = d.make(bad, 3);
  if (d.result()) return -1;
  hipLaunchKernelGGL(quotient_check_kernel, blocks(n), dim3(256), 0, 0, dx, dc, n, db);
  d.err = hipGetLastError();
  d.read(bad, db, 3);
  for (int q = 0; q < 3; q++) mismatches[q] = (long long)bad[q];
  return d.result();
}

int pmx_check_force_mult(const double* num, const double* dvds, long long n, double krad,
                         double alpha, double* out) {
  if (!num || !dvds || n <= 0 || !out) { set_error("bad argument"); return -1; }
  Const k{};
  k.krad = krad;
  k.alpharad = alpha;
  DeviceArrays d;
  const double *dn = d.make(num, n), *dd = d.make(dvds, n);
  double* o = d.make((const double*)nullptr, 4 * n);
  if (d.result()) return -1;
  hipLaunchKernelGGL(force_check_kernel, blocks(n), dim3(256), 0, 0, dn, dd, n, k, o);
  d.err = hipGetLastError();
  d.read(out, o, 4 * n);
  return d.result();
}

int pmx_check_cooling(const pmx_wind_desc* desc, int on_device, long long n, const double* rho,
                      const double* p, const double* xi, const double* dt, const double* pre,
                      double* rate, double* e, double* p_out, long long* calls, int* flags) {
  if (!desc || n <= 0 || !rho || !p || !xi || !dt || !rate || !e || !p_out || !calls || !flags) {
    set_error("bad argument");
    return -1;
  }
  const Const k = make_const(desc);
  if (!on_device) {
    const CoolCheck c = {rho, p, xi, dt, pre, rate, e, p_out, calls, flags};
    for (long long i = 0; i < n; i++) check_cell(k, desc->t_x, c, n, i);
    return 0;
  }
  DeviceArrays d;
  CoolCheck c;
  c.rho = d.make(rho, n);
  c.p = d.make(p, n);
  c.xi = d.make(xi, n);
  c.dt = d.make(dt, n);
  c.pre = pre ? d.make(pre, 5 * n) : nullptr;
  c.rate = d.make((const double*)nullptr, n);
  c.e = d.make((const double*)nullptr, 2 * n);
  c.p_out = d.make((const double*)nullptr, 2 * n);
  c.calls = d.make((const long long*)nullptr, 3 * n);
  c.flags = d.make((const int*)nullptr, n);
  if (d.result()) return -1;
  hipLaunchKernelGGL(cool_check_kernel, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, 0, k,
                     desc->t_x, c, n);
  d.err = hipGetLastError();
  d.read(rate, c.rate, n);
  d.read(e, c.e, 2 * n);
  d.read(p_out, c.p_out, 2 * n);
  d.read(calls, c.calls, 3 * n);
  d.read(flags, c.flags, n);
  return d.result();
}

}  // extern "C"
