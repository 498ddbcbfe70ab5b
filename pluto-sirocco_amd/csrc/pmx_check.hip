// Arithmetic check: the short operations of the plain cooling integrator
// beside the general ones, on the same cells.  It calls the functions the
// kernels call, from a translation unit of its own, so that the kernels'
// inlining does not depend on it.
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
