// libplutomx: hydro context, step driver and C ABI (see include/plutomx.h).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/plutomx.h"
#include "pmx_common.h"
#include "pmx_hydro_kernels.h"

namespace pmx {

static thread_local std::string g_err;
void set_error(const std::string& msg) { g_err = msg; }

// dt/dx for every cell and direction, and reset of the step reductions.
// A main-loop step (dt_override null) does nothing once the run has halted.
__global__ void prep_kernel(DevScalars* s, const double* dx, double* dtdx, int ntot,
                            const double* dt_override) {
  if (!dt_override && s->halt) return;
  double dt = dt_override ? *dt_override : s->dt;
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  for (int q = t; q < ntot; q += gridDim.x * blockDim.x) dtdx[q] = dt / dx[q];
  if (t < RED_SLOTS) s->cdt_red[red_index(t)] = 0ull;
  if (t == 0) {
    if (dt_override) s->dt = dt;
    s->err = 0;
  }
}

// The end of a step taken through the dt/dx table (3-D, or an explicit
// step): end_step, then, in the main loop while the run goes on, what
// prep_kernel would do for the next step: dt/dx with the next dt and the
// cleared C_dt slots (the next step's own prep launch is then left out).
__global__ __launch_bounds__(256) void finish_kernel(DevScalars* s, StepRule rule, int loop,
                                                     const double* inv_in, const double* dx,
                                                     double* dtdx, int ntot) {
  __shared__ int go;
  __shared__ double dt_next;
  StepState q = *s;
  const unsigned long long m = fold_cdt(s);
  __syncthreads();                     // every thread has read before one writes
  if (loop && q.halt) return;
  if (threadIdx.x == 0) {
    end_step(q, m, rule, loop, inv_in ? *inv_in : 0.0);
    static_cast<StepState&>(*s) = q;
    go = loop && !q.halt;
    dt_next = q.dt;
  }
  __syncthreads();
  if (!go) return;
  for (int q = threadIdx.x; q < ntot; q += blockDim.x) dtdx[q] = dt_next / dx[q];
  if (threadIdx.x < RED_SLOTS) s->cdt_red[red_index(threadIdx.x)] = 0ull;
}

// The end of a 2-D main-loop run: end_step on the last step's state
// s[which], the result in s[0], the reductions of both states cleared.
__global__ __launch_bounds__(64) void finish_run_kernel(DevScalars* s, int which, StepRule rule) {
  const unsigned long long m = fold_cdt(s + which);
  StepState q = s[which];
  if (q.pending && !q.halt) end_step(q, m, rule, 1, 0.0);
  __syncthreads();                     // every lane has read before any writes
  if (threadIdx.x == 0) {
    static_cast<StepState&>(s[0]) = q;
    s[1].err = 0;
  }
  const int k = threadIdx.x;
  s[k / RED_SLOTS].cdt_red[red_index(k % RED_SLOTS)] = 0ull;
}

// PLUTO's ghosted Vc[nv][k][j][i] from / to the interior arrays, the ghost
// cells filled by the boundary rules, and its Uc[cell][nv] from U: values
// q0 .. q0 + m of PLUTO's array from / to a buffer.  The host's transfers are
// then of arrays as PLUTO holds them; these passes take 10 us each (14 MB,
// 64^3) where loops over the host arrays took 3.8 ms of a 64^3
// step's download and 0.4 ms of its upload.
struct GhostLayout {
  int nx, ny, nz, g[3];          // interior, ghost cells per direction
  int bc[6];
  __host__ __device__ long long tx() const { return nx + 2 * g[0]; }
  __host__ __device__ long long ty() const { return ny + 2 * g[1]; }
  __host__ __device__ long long tz() const { return nz + 2 * g[2]; }
  __host__ __device__ long long cells() const { return tx() * ty() * tz(); }
};

// Variable and indices of value q of the ghosted array.  (A grid that fits
// the device has fewer than 2^32 cells: the divisions are 32-bit ones.)
struct GhostIndex {
  int nv, i, j, k;
};
__device__ __forceinline__ GhostIndex ghost_index(const GhostLayout& L, long long q) {
  GhostIndex x;
  const long long n = L.cells();
  x.nv = 0;
#pragma unroll
  for (int v = 1; v < NV; v++) {
    const bool past = q >= n;
    q -= past ? n : 0;
    x.nv += past;
  }
  const unsigned tx = (unsigned)L.tx(), ty = (unsigned)L.ty(), r = (unsigned)q, row = r / tx;
  x.i = (int)(r - row * tx);
  x.k = (int)(row / ty);
  x.j = (int)(row - x.k * ty);
  return x;
}

__global__ __launch_bounds__(256) void ghost_pack_kernel(const double* __restrict__ V,
                                                         double* __restrict__ buf, GhostLayout L,
                                                         long long q0, long long m) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= m) return;
  const GhostIndex x = ghost_index(L, q0 + q);
  bool flip[3] = {false, false, false};
  const int i = map_bc(x.i - L.g[0], L.nx, L.bc[0], L.bc[1], flip[0]);
  const int j = map_bc(x.j - L.g[1], L.ny, L.bc[2], L.bc[3], flip[1]);
  const int k = L.g[2] ? map_bc(x.k - L.g[2], L.nz, L.bc[4], L.bc[5], flip[2]) : 0;
  const double v = V[(((long long)x.nv * L.nz + k) * L.ny + j) * L.nx + i];
  const bool neg = (x.nv == VX1 && flip[0]) || (x.nv == VX2 && flip[1]) ||
                   (x.nv == VX3 && flip[2]);
  buf[q] = neg ? -v : v;
}

__global__ __launch_bounds__(256) void ghost_unpack_kernel(const double* __restrict__ buf,
                                                           double* __restrict__ V, GhostLayout L,
                                                           long long q0, long long m) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= m) return;
  const GhostIndex x = ghost_index(L, q0 + q);
  const int i = x.i - L.g[0], j = x.j - L.g[1], k = x.k - L.g[2];
  if (i >= 0 && i < L.nx && j >= 0 && j < L.ny && k >= 0 && k < L.nz)
    V[(((long long)x.nv * L.nz + k) * L.ny + j) * L.nx + i] = buf[q];
}

__global__ __launch_bounds__(256) void cons_interleave_kernel(const double* __restrict__ U,
                                                              double* __restrict__ buf,
                                                              long long ncell, long long q0,
                                                              long long m) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < m) buf[q] = U[(q0 + q) % NV * ncell + (q0 + q) / NV];
}

// Plain streaming copy, used to calibrate the HBM byte counters and to
// measure the bandwidth a simple kernel reaches on this device.
__global__ void copy_probe_kernel(const double2* __restrict__ src, double2* __restrict__ dst,
                                  long long n2) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long stride = (long long)gridDim.x * blockDim.x;
  for (long long q = t; q < n2; q += stride) dst[q] = src[q];
}

}  // namespace pmx

using namespace pmx;

struct pmx_hydro {
  pmx_hydro_desc d;
  int nx, ny, nz;
  long long ncell;
  double* V[3];
  double* U;
  double* dx;       // [nx | ny | nz]
  double* dtdx;
  double* inv_dl;
  DevScalars* s;    // the time state, and the other one of a 2-D run
  double* dt_in;    // device slots of an explicit step: dt, and Dts->invDt_hyp on entry
  hipStream_t stream;
  hipGraphExec_t graph;
  bool have_graph;
  bool timing;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> ev_pending;
  double timed_ms;
  int timed_launches;
  long long piece;  // values of PLUTO's arrays handed over at a time, through V[1]
};

namespace {

// The z chunks of a 3-D grid of `tiles` x-y tiles.
struct ZPlan {
  int n;                          // chunks of zc0, or 0: uniform chunks of cz planes
  int zc0[PMX_MAX_ZCHUNKS + 1];
  int cz;
};

// z chunks of decreasing length: `size` planes while more than 2 size
// remain, then half of that, ..., then pieces of `least` planes (nz = 256,
// 64 and 8: 64, 64, 32, 32, 16, 16, 8, 8, 8, 8), long ones dispatched
// first.  Returns the number of chunks, or 0 when they do not fit zc0.
int z_decreasing(int nz, int size, int least, int* zc0) {
  int n = 0, z = 0, rem = nz;
  auto push = [&](int len) { zc0[n++] = z; z += len; rem -= len; };
  for (; size >= least; size /= 2)
    while (rem > 2 * size && n < PMX_MAX_ZCHUNKS) push(size);
  while (rem > 0 && n < PMX_MAX_ZCHUNKS) push(rem < least ? rem : least);
  zc0[n] = nz;
  return rem == 0 ? n : 0;
}

// How the z planes are cut among workgroups.  256 CUs hold two workgroups
// each; a chunk of L planes costs a workgroup L + 1.45 plane times (the
// ghost planes, two states and a face of its start), a plane taking 8.3 us
// next to a second workgroup of the CU and 5.5 us alone (PPM + HLLC).  Two
// plans are priced that way and the cheaper one is taken:
//  * one round: equal chunks, as many as let every workgroup be resident
//    at once (or one per CU).  It suits grids of few tiles, whose launch
//    would otherwise last as long as its longest chunk: per stage 64^3
//    (20 tiles) takes 37 us in 3-plane chunks against 101 us in chunks of
//    16 .. 8, 101 x 66 x 93 (35 tiles) 73 us in 7-plane chunks against 193;
//  * chunks of decreasing length, the longest at most 7/16 of the planes a
//    slot gets: long chunks cost less in re-read ghost planes, the short
//    ones dispatched last let every CU finish together.  Sedov 256^3 (64 ..
//    8): 1.265 ms per stage, equal 16-plane chunks 1.311, 32-plane ones
//    1.354.
// PMX_CZ sets uniform chunks of its own.
ZPlan z_plan(int tiles, int nz) {
  ZPlan p;
  p.n = 0;
  p.cz = nz < 64 ? 8 : 16;
  if (const char* e = getenv("PMX_CZ")) {
    p.cz = atoi(e) > 0 ? atoi(e) : p.cz;
    return p;
  }
  const int cus = 256, slots = 2 * cus;
  const double start = 1.45, alone = 0.66;
  double best = 1e300;
  for (int fit : {slots, cus}) {
    const int n = std::min(fit / tiles, nz);
    if (n < 1) continue;
    const int len = (nz + n - 1) / n;
    const double t = (len + start) * (tiles * ((nz + len - 1) / len) <= cus ? alone : 1.0);
    if (t < best) { best = t; p.cz = len; }
  }
  const double share = (double)tiles * nz / slots;   // planes per slot
  int size = 64;
  while (size > 2 && size > share * 0.4375) size /= 2;
  const int least = std::min(8, std::max(2, size / 2));
  p.n = z_decreasing(nz, size, least, p.zc0);
  if (p.n == 0) {                  // a column too long for zc0
    if (best > 1e299) p.cz = size;
    return p;
  }
  // later rounds overlap the starts of their chunks with other workgroups'
  // planes: 0.6 planes per chunk, and 0.87 of the price of one round
  const double t = 0.87 * (tiles * (nz + 0.6 * p.n) / slots + 0.5 * (least + start));
  if (best <= t) p.n = 0;
  return p;
}

// The boundary kind of a domain: one rule on every side of the active
// directions is compiled in (BCK_OUTFLOW, BCK_PERIODIC), else BCK_ANY.
int boundary_kind(const pmx_hydro_desc& d) {
  const int ns = 2 * d.dims;
  bool out = true, per = true;
  for (int q = 0; q < ns; q++) {
    out = out && d.bc[q] == PMX_BC_OUTFLOW;
    per = per && d.bc[q] == PMX_BC_PERIODIC;
  }
  return out ? BCK_OUTFLOW : (per ? BCK_PERIODIC : BCK_ANY);
}

template <int DIMS, int REC, int SOLVER, int MODE>
void launch_stage(pmx_hydro* h, const StageArgs& a, int nblocks) {
  const dim3 g(nblocks), b(NTHREADS);
  const int bck = boundary_kind(h->d);
  if (bck == BCK_ANY) {   // mixed sides: compiled in pmx_hydro_any.hip
    launch_stage_any(DIMS, REC, SOLVER, MODE, a, nblocks, h->stream);
    return;
  }
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, 0, h->stream, a); };
  auto by_bck = [&](auto ty) {
    constexpr int TY = decltype(ty)::value;
    if (bck == BCK_OUTFLOW)
      launch(stage_kernel<DIMS, REC, SOLVER, MODE, BCK_OUTFLOW, TILE_X, TY, NTHREADS>);
    else
      launch(stage_kernel<DIMS, REC, SOLVER, MODE, BCK_PERIODIC, TILE_X, TY, NTHREADS>);
  };
  if constexpr (DIMS == 2) {
    if (a.tile_y == TILE_Y_2D) {
      by_bck(std::integral_constant<int, TILE_Y_2D>());
      return;
    }
  }
  by_bck(std::integral_constant<int, TILE_Y>());
}

template <int DIMS, int REC, int SOLVER>
void dispatch_mode(pmx_hydro* h, const StageArgs& a, int nblocks, int mode) {
  if (mode == MODE_FIRST) launch_stage<DIMS, REC, SOLVER, MODE_FIRST>(h, a, nblocks);
  else if (mode == MODE_WEIGHTED) launch_stage<DIMS, REC, SOLVER, MODE_WEIGHTED>(h, a, nblocks);
  else launch_stage<DIMS, REC, SOLVER, MODE_THIRD>(h, a, nblocks);
}

template <int DIMS, int REC>
void dispatch_solver(pmx_hydro* h, const StageArgs& a, int nblocks, int mode) {
  if (h->d.solver == PMX_SOLVER_ROE) dispatch_mode<DIMS, REC, SOL_ROE>(h, a, nblocks, mode);
  else dispatch_mode<DIMS, REC, SOL_HLLC>(h, a, nblocks, mode);
}

template <int DIMS>
void dispatch_rec(pmx_hydro* h, const StageArgs& a, int nblocks, int mode) {
  switch (h->d.recon) {
    case PMX_REC_PLM_VANLEER: dispatch_solver<DIMS, REC_PLM_VL>(h, a, nblocks, mode); break;
    case PMX_REC_PLM_MC: dispatch_solver<DIMS, REC_PLM_MC>(h, a, nblocks, mode); break;
    case PMX_REC_PLM_MINMOD: dispatch_solver<DIMS, REC_PLM_MM>(h, a, nblocks, mode); break;
    case PMX_REC_PLM_DEFAULT: dispatch_solver<DIMS, REC_PLM_DEFAULT>(h, a, nblocks, mode); break;
    default: dispatch_solver<DIMS, REC_PPM>(h, a, nblocks, mode); break;
  }
}

StepRule step_rule(const pmx_hydro* h) {
  return {h->d.dims, h->d.cfl, h->d.cfl_max_var, h->d.first_dt};
}

// cur: the step's time state; prev: the previous step's (2-D main-loop
// stages 1 and 2), or null.
int stage(pmx_hydro* h, const double* Vin, const double* V0, double* Vout, int mode, double w0,
          double wc, int write_u, bool loop, DevScalars* cur, DevScalars* prev) {
  StageArgs a;
  a.Vin = Vin;
  a.V0 = V0;
  a.U = h->U;
  a.Vout = Vout;
  a.nx = h->nx; a.ny = h->ny; a.nz = h->nz;
  a.sv = h->ncell;
  for (int q = 0; q < 6; q++) a.bc[q] = h->d.bc[q];
  a.gamma = h->d.gamma;
  a.gmm1 = h->d.gamma - 1.0;
  a.rg = recip2(a.gmm1, 1.0 / a.gmm1);
  a.dtdx[0] = h->dtdx; a.dtdx[1] = h->dtdx + h->nx; a.dtdx[2] = h->dtdx + h->nx + h->ny;
  a.inv_dl[0] = h->inv_dl; a.inv_dl[1] = h->inv_dl + h->nx; a.inv_dl[2] = h->inv_dl + h->nx + h->ny;
  a.w0 = w0; a.wc = wc;
  a.tiles_x = (h->nx + TILE_X - 1) / TILE_X;
  a.tile_y = tile_height(h->d.dims, h->nx, h->ny);
  a.tiles_y = (h->ny + a.tile_y - 1) / a.tile_y;
  a.nzc = 0;
  a.cz = 1;
  a.tiles_z = 1;
  if (h->d.dims == 3) {
    const ZPlan p = z_plan(a.tiles_x * a.tiles_y, h->nz);
    a.nzc = p.n;
    if (p.n) memcpy(a.zc0, p.zc0, sizeof(int) * (p.n + 1));
    a.cz = p.cz;
    a.tiles_z = p.n ? p.n : (h->nz + p.cz - 1) / p.cz;
  }
  a.write_u = write_u;
  a.cdt_bits = cur->cdt_red;
  a.err = &cur->err;
  // (stage 1 of a 2-D main-loop step sets cur->halt itself)
  a.halt = loop && !(prev && mode == MODE_FIRST) ? &cur->halt : nullptr;
  a.dx[0] = h->dx;
  a.dx[1] = h->dx + h->nx;
  a.cur = cur;
  a.prev = prev;
  a.rule = step_rule(h);
  // with the z schedule, 8 ceil(tiles / 8) workgroups per chunk (a whole
  // number per XCD; see stage_kernel)
  int nblocks = a.nzc ? 8 * ((a.tiles_x * a.tiles_y + 7) / 8) * a.nzc
                      : a.tiles_x * a.tiles_y * a.tiles_z;

  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (h->timing) {
    if (h->ev_pool.size() < 2) {
      for (int q = 0; q < 64; q++) {
        hipEvent_t e;
        PMX_HIP_CHECK(hipEventCreate(&e));
        h->ev_pool.push_back(e);
      }
    }
    e0 = h->ev_pool.back(); h->ev_pool.pop_back();
    e1 = h->ev_pool.back(); h->ev_pool.pop_back();
    PMX_HIP_CHECK(hipEventRecord(e0, h->stream));
  }
  if (h->d.dims == 3) dispatch_rec<3>(h, a, nblocks, mode);
  else dispatch_rec<2>(h, a, nblocks, mode);
  PMX_HIP_CHECK(hipGetLastError());
  if (h->timing) {
    PMX_HIP_CHECK(hipEventRecord(e1, h->stream));
    h->ev_pending.push_back({e0, e1});
  }
  return 0;
}

// The RK stages of one AdvanceStep: Src/Time_Stepping/rk_step.c:117-330.
// V[0] holds V^n on entry and V^{n+1} on exit.
int stages(pmx_hydro* h, bool loop, DevScalars* cur, DevScalars* prev) {
  if (h->d.rk == 3) {
    if (stage(h, h->V[0], h->V[0], h->V[1], MODE_FIRST, 0, 0, 1, loop, cur, prev)) return -1;
    if (stage(h, h->V[1], h->V[0], h->V[2], MODE_WEIGHTED, 0.75, 0.25, 1, loop, cur, prev))
      return -1;
    return stage(h, h->V[2], h->V[0], h->V[0], MODE_THIRD, 0, 0, 1, loop, cur, nullptr);
  }
  if (stage(h, h->V[0], h->V[0], h->V[1], MODE_FIRST, 0, 0, 1, loop, cur, prev)) return -1;
  return stage(h, h->V[1], h->V[0], h->V[0], MODE_WEIGHTED, 0.5, 0.5, 1, loop, cur, prev);
}

// One step through the dt/dx table.  In the main loop (dt_override null)
// the previous step's finish_kernel has prepared this one (dt/dx, cleared
// slots) unless the run is just starting (with_prep).
int advance(pmx_hydro* h, const double* dt_override, bool with_prep) {
  int ntot = h->nx + h->ny + h->nz;
  const bool loop = dt_override == nullptr;
  if (with_prep || !loop) {
    hipLaunchKernelGGL(prep_kernel, dim3((ntot + 255) / 256), dim3(256), 0, h->stream, h->s,
                       h->dx, h->dtdx, ntot, dt_override);
    PMX_HIP_CHECK(hipGetLastError());
  }
  if (stages(h, loop, h->s, nullptr)) return -1;
  hipLaunchKernelGGL(finish_kernel, dim3(1), dim3(256), 0, h->stream, h->s, step_rule(h),
                     loop ? 1 : 0, loop ? nullptr : dt_override + 1, h->dx, h->dtdx, ntot);
  PMX_HIP_CHECK(hipGetLastError());
  return 0;
}

// Steps first .. first + n - 1 of a main-loop run.  A 2-D step is its stage
// kernels alone: the time state alternates between s[0] and s[1], each
// step's stage 1 ending the one before (KH 64^2: 17.6 -> 13.4 us per step, with
// three runs side by side on streams of their own 6.4 -> 4.9).
int run_steps(pmx_hydro* h, int first, int n) {
  for (int q = first; q < first + n; q++) {
    if (h->d.dims == 2) {
      if (stages(h, true, h->s + (q + 1) % 2, h->s + q % 2)) return -1;
    } else if (advance(h, nullptr, q == 0)) {
      return -1;
    }
  }
  return 0;
}

// After nsteps main-loop steps: the 2-D run's time state back in s[0].
int end_run(pmx_hydro* h, int nsteps) {
  if (h->d.dims != 2 || nsteps == 0) return 0;
  hipLaunchKernelGGL(finish_run_kernel, dim3(1), dim3(64), 0, h->stream, h->s, nsteps % 2,
                     step_rule(h));
  PMX_HIP_CHECK(hipGetLastError());
  return 0;
}

int collect_timing(pmx_hydro* h) {
  for (auto& p : h->ev_pending) {
    float ms = 0.f;
    PMX_HIP_CHECK(hipEventSynchronize(p.second));
    PMX_HIP_CHECK(hipEventElapsedTime(&ms, p.first, p.second));
    h->timed_ms += ms;
    h->timed_launches++;
    h->ev_pool.push_back(p.first);
    h->ev_pool.push_back(p.second);
  }
  h->ev_pending.clear();
  return 0;
}

GhostLayout ghost_layout(const pmx_hydro* h) {
  GhostLayout L;
  L.nx = h->nx; L.ny = h->ny; L.nz = h->nz;
  const int ng = h->d.recon == PMX_REC_PPM ? 3 : 2;
  L.g[0] = L.g[1] = ng;
  L.g[2] = h->d.dims == 3 ? ng : 0;
  for (int q = 0; q < 6; q++) L.bc[q] = h->d.bc[q];
  return L;
}

// PLUTO's arrays are handed over in pieces through V[1], which holds nothing
// between two steps, so a hand-over needs no memory of its own.  V[1] is made
// long enough that a ghosted array of up to HANDOVER_MIN values goes in one
// piece (64^3: 1.7 M values, a step with both transfers 2.07 ms); a piece is
// at most HANDOVER_MAX values, a launch of one thread each.
constexpr long long HANDOVER_MIN = 1ll << 22, HANDOVER_MAX = 1ll << 28;

long long handover_values(const pmx_hydro* h) {
  return std::max(NV * h->ncell, std::min(NV * ghost_layout(h).cells(), HANDOVER_MIN));
}

unsigned blocks256(long long n) { return (unsigned)((n + 255) / 256); }

// f(q0, m) for the pieces of an array of n values
template <class F>
int by_pieces(const pmx_hydro* h, long long n, F f) {
  for (long long q0 = 0; q0 < n; q0 += h->piece)
    if (f(q0, std::min(h->piece, n - q0))) return -1;
  return 0;
}

// The checks pmx_hydro_create makes of a descriptor.
int check_desc(const pmx_hydro_desc* desc) {
  if (desc->dims != 2 && desc->dims != 3) { set_error("dims must be 2 or 3"); return -1; }
  if (desc->rk != 2 && desc->rk != 3) { set_error("rk must be 2 or 3"); return -1; }
  if (desc->recon != PMX_REC_PLM_VANLEER && desc->recon != PMX_REC_PLM_MC &&
      desc->recon != PMX_REC_PLM_MINMOD && desc->recon != PMX_REC_PLM_DEFAULT &&
      desc->recon != PMX_REC_PPM) {
    set_error("unknown reconstruction"); return -1;
  }
  if (desc->solver != PMX_SOLVER_HLLC && desc->solver != PMX_SOLVER_ROE) {
    set_error("unknown Riemann solver"); return -1;
  }
  for (int q = 0; q < 6; q++)
    if (desc->bc[q] < 0 || desc->bc[q] > 2) { set_error("unknown boundary type"); return -1; }
  int nz = desc->dims == 3 ? desc->nx3 : 1;
  int H = desc->recon == PMX_REC_PPM ? 3 : 2;
  if (desc->nx1 < H || desc->nx2 < H || (desc->dims == 3 && desc->nx3 < H)) {
    set_error("grid smaller than the ghost width"); return -1;
  }
  if (!desc->dx1 || !desc->dx2 || (desc->dims == 3 && !desc->dx3)) {
    set_error("missing cell widths"); return -1;
  }
  return 0;
}

// dx per cell of every direction ([nx | ny | nz]) and its reciprocal
// (Src/set_geometry.c:305).
void host_tables(const pmx_hydro_desc* desc, int nx, int ny, int nz, std::vector<double>& dx,
                 std::vector<double>& inv) {
  const int ntot = nx + ny + nz;
  dx.resize(ntot);
  inv.resize(ntot);
  for (int i = 0; i < nx; i++) dx[i] = desc->dx1[i];
  for (int j = 0; j < ny; j++) dx[nx + j] = desc->dx2[j];
  for (int k = 0; k < nz; k++) dx[nx + ny + k] = desc->dims == 3 ? desc->dx3[k] : 1.0;
  for (int q = 0; q < ntot; q++) inv[q] = 1.0 / dx[q];
}

}  // namespace

extern "C" {

const char* pmx_last_error(void) { return g_err.c_str(); }

int pmx_hydro_create(const pmx_hydro_desc* desc, pmx_hydro** out) {
  if (!desc || !out) { set_error("null argument"); return -1; }
  if (check_desc(desc)) return -1;
  int nz = desc->dims == 3 ? desc->nx3 : 1;
  pmx_hydro* h = new pmx_hydro();
  h->d = *desc;
  h->nx = desc->nx1; h->ny = desc->nx2; h->nz = nz;
  h->ncell = (long long)h->nx * h->ny * h->nz;
  size_t vbytes = sizeof(double) * NV * h->ncell;
  int ntot = h->nx + h->ny + h->nz;
#define CK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { \
    set_error(std::string(#x) + ": " + hipGetErrorString(e_)); pmx_hydro_destroy(h); return -1; } } while (0)
  CK(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  const long long held = handover_values(h);
  h->piece = std::min(held, HANDOVER_MAX);
  for (int q = 0; q < 3; q++) CK(hipMalloc(&h->V[q], q == 1 ? sizeof(double) * held : vbytes));
  CK(hipMalloc(&h->U, vbytes));
  CK(hipMalloc(&h->dx, sizeof(double) * ntot));
  CK(hipMalloc(&h->dtdx, sizeof(double) * ntot));
  CK(hipMalloc(&h->inv_dl, sizeof(double) * ntot));
  CK(hipMalloc(&h->s, 2 * sizeof(DevScalars)));
  CK(hipMalloc(&h->dt_in, 2 * sizeof(double)));
  {
    std::vector<double> dx, inv;
    host_tables(desc, h->nx, h->ny, h->nz, dx, inv);
    CK(hipMemcpy(h->dx, dx.data(), sizeof(double) * ntot, hipMemcpyHostToDevice));
    CK(hipMemcpy(h->inv_dl, inv.data(), sizeof(double) * ntot, hipMemcpyHostToDevice));
    DevScalars s0[2] = {};
    s0[0].tstop = HUGE_VAL;
    CK(hipMemcpy(h->s, s0, sizeof(s0), hipMemcpyHostToDevice));
  }
  for (int q = 0; q < 3; q++) CK(hipMemset(h->V[q], 0, vbytes));
  CK(hipMemset(h->U, 0, vbytes));
#undef CK
  *out = h;
  return 0;
}

int pmx_hydro_destroy(pmx_hydro* h) {
  if (!h) return 0;
  if (h->stream) hipStreamSynchronize(h->stream);
  if (h->have_graph) hipGraphExecDestroy(h->graph);
  for (auto& p : h->ev_pending) { h->ev_pool.push_back(p.first); h->ev_pool.push_back(p.second); }
  for (auto e : h->ev_pool) hipEventDestroy(e);
  for (int q = 0; q < 3; q++) if (h->V[q]) hipFree(h->V[q]);
  if (h->U) hipFree(h->U);
  if (h->dx) hipFree(h->dx);
  if (h->dtdx) hipFree(h->dtdx);
  if (h->inv_dl) hipFree(h->inv_dl);
  if (h->s) hipFree(h->s);
  if (h->dt_in) hipFree(h->dt_in);
  if (h->stream) hipStreamDestroy(h->stream);
  delete h;
  return 0;
}

int pmx_hydro_set_prim(pmx_hydro* h, const double* V, int ghosts) {
  if (!h || !V) { set_error("null argument"); return -1; }
  if (ghosts) {
    const GhostLayout L = ghost_layout(h);
    if (by_pieces(h, NV * L.cells(), [&](long long q0, long long m) {
          PMX_HIP_CHECK(hipMemcpyAsync(h->V[1], V + q0, m * sizeof(double), hipMemcpyHostToDevice,
                                       h->stream));
          hipLaunchKernelGGL(ghost_unpack_kernel, dim3(blocks256(m)), dim3(256), 0, h->stream,
                             h->V[1], h->V[0], L, q0, m);
          PMX_HIP_CHECK(hipGetLastError());
          return 0;
        })) return -1;
  } else {
    PMX_HIP_CHECK(hipMemcpyAsync(h->V[0], V, sizeof(double) * NV * h->ncell,
                                 hipMemcpyHostToDevice, h->stream));
  }
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  return 0;
}

int pmx_hydro_get_prim(pmx_hydro* h, double* V, int ghosts) {
  if (!h || !V) { set_error("null argument"); return -1; }
  if (ghosts) {
    const GhostLayout L = ghost_layout(h);
    if (by_pieces(h, NV * L.cells(), [&](long long q0, long long m) {
          hipLaunchKernelGGL(ghost_pack_kernel, dim3(blocks256(m)), dim3(256), 0, h->stream,
                             h->V[0], h->V[1], L, q0, m);
          PMX_HIP_CHECK(hipGetLastError());
          PMX_HIP_CHECK(hipMemcpyAsync(V + q0, h->V[1], m * sizeof(double),
                                       hipMemcpyDeviceToHost, h->stream));
          return 0;
        })) return -1;
  } else {
    PMX_HIP_CHECK(hipMemcpyAsync(V, h->V[0], sizeof(double) * NV * h->ncell,
                                 hipMemcpyDeviceToHost, h->stream));
  }
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  return 0;
}

int pmx_hydro_get_cons(pmx_hydro* h, double* U, int pluto_layout) {
  if (!h || !U) { set_error("null argument"); return -1; }
  if (pluto_layout) {
    if (by_pieces(h, NV * h->ncell, [&](long long q0, long long m) {
          hipLaunchKernelGGL(cons_interleave_kernel, dim3(blocks256(m)), dim3(256), 0, h->stream,
                             h->U, h->V[1], h->ncell, q0, m);
          PMX_HIP_CHECK(hipGetLastError());
          PMX_HIP_CHECK(hipMemcpyAsync(U + q0, h->V[1], m * sizeof(double),
                                       hipMemcpyDeviceToHost, h->stream));
          return 0;
        })) return -1;
  } else {
    PMX_HIP_CHECK(hipMemcpyAsync(U, h->U, sizeof(double) * NV * h->ncell, hipMemcpyDeviceToHost,
                                 h->stream));
  }
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  return 0;
}

int pmx_hydro_set_time(pmx_hydro* h, double t, double dt) {
  if (!h) { set_error("null argument"); return -1; }
  DevScalars s0;
  PMX_HIP_CHECK(hipMemcpyAsync(&s0, h->s, sizeof(s0), hipMemcpyDeviceToHost, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  s0.t = t;
  s0.dt = dt;
  s0.halt = 0;
  s0.last = 0;
  clamp_last_step(s0);
  PMX_HIP_CHECK(hipMemcpyAsync(h->s, &s0, sizeof(s0), hipMemcpyHostToDevice, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  return 0;
}

int pmx_hydro_set_tstop(pmx_hydro* h, double tstop) {
  if (!h || !(tstop > -HUGE_VAL)) { set_error("bad argument"); return -1; }
  DevScalars s0;
  PMX_HIP_CHECK(hipMemcpyAsync(&s0, h->s, sizeof(s0), hipMemcpyDeviceToHost, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  s0.tstop = tstop;
  s0.halt &= ~PMX_FLAG_TSTOP;
  if (s0.last) {           // undo a cut made for the previous tstop
    s0.dt = s0.dt_uncut;
    s0.last = 0;
  }
  clamp_last_step(s0);
  PMX_HIP_CHECK(hipMemcpyAsync(h->s, &s0, sizeof(s0), hipMemcpyHostToDevice, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  return 0;
}

int pmx_hydro_get_time(pmx_hydro* h, double* t, double* dt, double* inv_dt_hyp, int* flags) {
  if (!h) { set_error("null argument"); return -1; }
  DevScalars s0;
  PMX_HIP_CHECK(hipMemcpyAsync(&s0, h->s, sizeof(s0), hipMemcpyDeviceToHost, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  if (t) *t = s0.t;
  if (dt) *dt = s0.dt;
  if (inv_dt_hyp) *inv_dt_hyp = s0.inv_dt_hyp;
  if (flags) *flags = s0.step_err | s0.err | s0.halt;
  return 0;
}

int pmx_hydro_advance_step(pmx_hydro* h, double dt, double* inv_dt_hyp) {
  if (!h) { set_error("null argument"); return -1; }
  const double in[2] = {dt, inv_dt_hyp ? *inv_dt_hyp : 0.0};
  PMX_HIP_CHECK(hipMemcpyAsync(h->dt_in, in, sizeof(in), hipMemcpyHostToDevice, h->stream));
  if (advance(h, h->dt_in, true)) return -1;
  if (h->timing) collect_timing(h);
  DevScalars s0;
  PMX_HIP_CHECK(hipMemcpyAsync(&s0, h->s, sizeof(s0), hipMemcpyDeviceToHost, h->stream));
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  if (inv_dt_hyp) *inv_dt_hyp = s0.inv_dt_hyp;
  return 0;
}

int pmx_hydro_run(pmx_hydro* h, int nsteps) {
  if (!h || nsteps < 0) { set_error("bad argument"); return -1; }
  return run_steps(h, 0, nsteps) || end_run(h, nsteps) ? -1 : 0;
}

// Steps per captured graph (an even number, so that a 2-D graph ends where
// it began, in s[0]): a graph launch costs more than the few kernel
// launches of one step saves (KH 256^2: 33 us per step replaying one step
// per graph against 26 us eager), so a graph holds several steps.  Steps
// after the run halts are no-ops on the device, as in the eager loop.
constexpr int GRAPH_STEPS = 8;

int pmx_hydro_run_graph(pmx_hydro* h, int nsteps) {
  if (!h || nsteps < 0) { set_error("bad argument"); return -1; }
  if (h->timing) return pmx_hydro_run(h, nsteps);
  if (nsteps >= GRAPH_STEPS && !h->have_graph) {
    hipGraph_t g;
    PMX_HIP_CHECK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    const int rc = run_steps(h, 0, GRAPH_STEPS);
    hipError_t e = hipStreamEndCapture(h->stream, &g);
    if (rc) return -1;
    if (e != hipSuccess) { set_error(std::string("capture: ") + hipGetErrorString(e)); return -1; }
    PMX_HIP_CHECK(hipGraphInstantiate(&h->graph, g, nullptr, nullptr, 0));
    PMX_HIP_CHECK(hipGraphDestroy(g));
    h->have_graph = true;
  }
  int n = 0;
  for (; nsteps - n >= GRAPH_STEPS; n += GRAPH_STEPS)
    PMX_HIP_CHECK(hipGraphLaunch(h->graph, h->stream));
  if (n < nsteps) {
    // (a 3-D remainder starts with its own prep launch, as step 0 does)
    if (run_steps(h, 0, nsteps - n)) return -1;
  }
  return end_run(h, nsteps);
}

int pmx_hydro_sync(pmx_hydro* h) {
  if (!h) { set_error("null argument"); return -1; }
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  if (h->timing) collect_timing(h);
  return 0;
}

int pmx_hydro_stage_timing(pmx_hydro* h, int enable, int reset, double* total_ms, int* launches) {
  if (!h) { set_error("null argument"); return -1; }
  PMX_HIP_CHECK(hipStreamSynchronize(h->stream));
  collect_timing(h);
  if (total_ms) *total_ms = h->timed_ms;
  if (launches) *launches = h->timed_launches;
  if (reset) { h->timed_ms = 0.0; h->timed_launches = 0; }
  h->timing = enable != 0;
  return 0;
}

// ---------------------------------------------------------------------
// The step without allocation: pmx_hydro_advance_step for callers that
// cannot allocate device memory (code under HIP graph capture, tight
// serving loops, harnesses that forbid hipMalloc).  The caller passes the
// state; everything else the step needs (the intermediate stage states,
// the dt/dx tables, the time scalars) lives in `scratch`, a fixed array
// in device memory that every GPU holds for the life of the process.
// ---------------------------------------------------------------------
}  // extern "C"

namespace {

constexpr long long NOALLOC_MAX_CELLS = 1ll << 19;   // 2 stage states of 5 doubles
constexpr int NOALLOC_MAX_LINE = 8192;               // nx + ny + nz
constexpr size_t NOALLOC_SCALARS = 16 + RED_SLOTS * RED_STRIDE;   // doubles for DevScalars
// [V1 | V2] stage states, then dx, dt/dx, 1/dx tables, the dt slots and
// the time scalars (with their spread reduction words): 40 MiB + 196 KiB
constexpr size_t NOALLOC_DOUBLES = 2 * (size_t)NV * NOALLOC_MAX_CELLS +
                                   3 * (size_t)NOALLOC_MAX_LINE + 2 + NOALLOC_SCALARS;
static_assert(sizeof(DevScalars) <= NOALLOC_SCALARS * sizeof(double), "scalar slots");

__device__ __align__(256) double scratch[NOALLOC_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
double* g_scratch[NOALLOC_MAX_DEVICES];   // scratch's address on each device, once looked up

// scratch's device address on the current device (host code never passes
// the array's name itself to a kernel: on the host it is a stand-in).
int noalloc_scratch(double** out) {
  int dev = 0;
  PMX_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) { set_error("device index out of range"); return -1; }
  if (!g_scratch[dev]) {
    void* p = nullptr;
    PMX_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[dev] = static_cast<double*>(p);
  }
  *out = g_scratch[dev];
  return 0;
}

}  // namespace

extern "C" {

int pmx_hydro_advance_step_noalloc(const pmx_hydro_desc* desc, double* V, double* U, double dt,
                                   double* inv_dt_hyp) {
  if (!desc || !V || !U) { set_error("null argument"); return -1; }
  if (check_desc(desc)) return -1;
  const int nx = desc->nx1, ny = desc->nx2, nz = desc->dims == 3 ? desc->nx3 : 1;
  const long long ncell = (long long)nx * ny * nz;
  if (ncell > NOALLOC_MAX_CELLS || nx + ny + nz > NOALLOC_MAX_LINE) {
    set_error("pmx_hydro_advance_step_noalloc: the grid (" + std::to_string(ncell) +
              " cells, nx+ny+nz = " + std::to_string(nx + ny + nz) + ") exceeds the limit of " +
              std::to_string(NOALLOC_MAX_CELLS) + " cells and nx+ny+nz <= " +
              std::to_string(NOALLOC_MAX_LINE) + " (use pmx_hydro_create)");
    return -1;
  }
  double* base = nullptr;
  if (noalloc_scratch(&base)) return -1;
  // a context on the stack whose device buffers are the caller's state and
  // slices of scratch; the step runs on the null stream and is waited for
  pmx_hydro h;
  h.d = *desc;
  h.nx = nx; h.ny = ny; h.nz = nz;
  h.ncell = ncell;
  h.V[0] = V;
  h.V[1] = base;
  h.V[2] = base + (size_t)NV * ncell;
  h.U = U;
  double* tab = base + 2 * (size_t)NV * NOALLOC_MAX_CELLS;
  const int ntot = nx + ny + nz;
  h.dx = tab;
  h.dtdx = tab + ntot;
  h.inv_dl = tab + 2 * ntot;
  h.dt_in = tab + 3 * NOALLOC_MAX_LINE;
  h.s = reinterpret_cast<DevScalars*>(h.dt_in + 2);
  h.stream = nullptr;
  h.have_graph = false;
  h.timing = false;
  h.timed_ms = 0.0;
  h.timed_launches = 0;
  std::vector<double> dx, inv;
  host_tables(desc, nx, ny, nz, dx, inv);
  DevScalars s0;
  s0 = DevScalars{};                // what the last call left is cleared
  s0.tstop = HUGE_VAL;
  const double in[2] = {dt, inv_dt_hyp ? *inv_dt_hyp : 0.0};
  PMX_HIP_CHECK(hipMemcpyAsync(h.dx, dx.data(), sizeof(double) * ntot, hipMemcpyHostToDevice, 0));
  PMX_HIP_CHECK(hipMemcpyAsync(h.inv_dl, inv.data(), sizeof(double) * ntot,
                               hipMemcpyHostToDevice, 0));
  PMX_HIP_CHECK(hipMemcpyAsync(h.s, &s0, sizeof(s0), hipMemcpyHostToDevice, 0));
  PMX_HIP_CHECK(hipMemcpyAsync(h.dt_in, in, sizeof(in), hipMemcpyHostToDevice, 0));
  if (advance(&h, h.dt_in, true)) return -1;
  PMX_HIP_CHECK(hipMemcpyAsync(&s0, h.s, sizeof(s0), hipMemcpyDeviceToHost, 0));
  PMX_HIP_CHECK(hipStreamSynchronize(0));
  if (inv_dt_hyp) *inv_dt_hyp = s0.inv_dt_hyp;
  return 0;
}

int pmx_copy_probe(long long nbytes, int reps, double* ms_per_copy) {
  if (nbytes <= 0 || nbytes % 16 != 0 || reps <= 0) { set_error("bad argument"); return -1; }
  double2 *a = nullptr, *b = nullptr;
  hipEvent_t e0, e1;
  PMX_HIP_CHECK(hipMalloc(&a, nbytes));
  if (hipMalloc(&b, nbytes) != hipSuccess) { hipFree(a); set_error("hipMalloc"); return -1; }
  hipMemset(a, 0, nbytes);
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  long long n2 = nbytes / 16;
  // 1024 workgroups of 256 threads striding over the buffer: the best of a
  // sweep of grid sizes (1024 .. 65536 workgroups) and per-thread unrolling
  // (1 .. 8 loads in flight) on MI355X, ~5.5 TB/s for 2 GiB
  hipLaunchKernelGGL(copy_probe_kernel, dim3(1024), dim3(256), 0, 0, a, b, n2);
  hipEventRecord(e0, 0);
  for (int r = 0; r < reps; r++)
    hipLaunchKernelGGL(copy_probe_kernel, dim3(1024), dim3(256), 0, 0, a, b, n2);
  hipEventRecord(e1, 0);
  hipError_t err = hipEventSynchronize(e1);
  float ms = 0.f;
  hipEventElapsedTime(&ms, e0, e1);
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  hipFree(a);
  hipFree(b);
  if (err != hipSuccess) { set_error(hipGetErrorString(err)); return -1; }
  if (ms_per_copy) *ms_per_copy = ms / reps;
  return 0;
}

int pmx_copy_probe_runtime(long long nbytes, int reps, double* ms_per_copy) {
  if (nbytes <= 0 || reps <= 0) { set_error("bad argument"); return -1; }
  void *a = nullptr, *b = nullptr;
  hipEvent_t e0, e1;
  PMX_HIP_CHECK(hipMalloc(&a, nbytes));
  if (hipMalloc(&b, nbytes) != hipSuccess) { hipFree(a); set_error("hipMalloc"); return -1; }
  hipMemset(a, 0, nbytes);
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  hipError_t err = hipMemcpyAsync(b, a, nbytes, hipMemcpyDeviceToDevice, 0);
  if (err == hipSuccess) err = hipEventRecord(e0, 0);
  for (int r = 0; r < reps && err == hipSuccess; r++)
    err = hipMemcpyAsync(b, a, nbytes, hipMemcpyDeviceToDevice, 0);
  if (err == hipSuccess) err = hipEventRecord(e1, 0);
  if (err == hipSuccess) err = hipEventSynchronize(e1);
  float ms = 0.f;
  if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  hipFree(a);
  hipFree(b);
  if (err != hipSuccess) { set_error(hipGetErrorString(err)); return -1; }
  if (ms_per_copy) *ms_per_copy = ms / reps;
  return 0;
}

int pmx_hydro_device_state(pmx_hydro* h, double** V, double** U) {
  if (!h) { set_error("null argument"); return -1; }
  if (V) *V = h->V[0];
  if (U) *U = h->U;
  return 0;
}

}  // extern "C"
