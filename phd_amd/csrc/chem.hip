// chem.hip -- batched stiff chemistry for CDNA4: CHEMKIN-form kinetics and a
// variable-order BDF integrator with Newton iteration and dense LU, run as a
// persistent kernel over a device work queue.
//
// Reference path replaced: reaction_dvode (devel-izem/src/module_reaction.f90:
// 102-304) -> PSR_CHEMKIN (chemkin/psr_chemkin.f:1-44) -> REACTION_V
// (chemkin/reaction_v.f:1-65: MF = 22, ITOL = 1, ITASK = 1, 20 restarts) ->
// DVODE (chemkin/vode.f:4286) -> FUN (reaction_v.f:69-114) -> CKWYR
// (vode.f:1797).  The integrator is this project's own implementation of
// the Nordsieck-form BDF method (orders 1-5, fixed-leading-coefficient
// rescaling on step changes, chord Newton with a Jacobian in closed form or
// by finite differences, weighted RMS error control); it agrees with DVODE to within the
// integration tolerance, not bit for bit.
#include "izem_ctx.h"

#include <limits.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "chem_tables.h"
#include "chem_setup.h"

__constant__ IzMech c_mech;
__constant__ IzBdf c_bdf;

#include "mech_gen.h"
#include "chem_device.h"

// bins of the stiffness key of izem_psr_batch: eight per octave of
// max_k |df_k/dY_k| [1/s] over [1, 2^64)
#define IZ_ORDER_BINS 512

struct IzChem {
  double rtol, atol;
  int trim;
  int *counter;     // work queue head
  int *istate;      // per-batch scratch for reaction_dvode
  // autotuned: register budget (waves per SIMD the kernel is compiled
  // for: 1, 2 or 4), resident 64-lane blocks per CU, Jacobian reuse age
  int waves, blocks_per_cu, jac_age;
  // the straight-line forms (mech_gen.h) that may run: bit f - 1 set where
  // the loaded mechanism is the compiled-in one and form f passed the check
  int generated;
  // work counters of the integrations since the last izem_chem_stats:
  // BDF steps, RHS evaluations, Jacobians, LU solves
  unsigned long long *stats;
  int use_gen;    // 0 tables, 1 straight-line kinetics, 2 with the closed-form Jacobian
  // stiffness order of izem_psr_batch: on/off, per-cell bin and queue
  // permutation (capacity order_cap cells), bin counts then offsets
  int order;
  long order_cap;
  int *order_bin, *order_perm, *order_hist;
  long order_n;   // cells of the last sorted batch, 0 when the last call ran unsorted
  // reaction_selec's solver (0 BDF, 1 surrogate with BDF fallback), the
  // attached surrogate, and a generation count of both for the step graph
  int reac_selec;
  struct IzSurr *surr;
  int sel_gen;
};

// a surrogate attached to the flow's reaction step: the caller's network
// and its workspace (feature rows and outputs of one chunk of cells, the
// list of fallback cells of the whole reacting box)
struct IzSurr {
  izem_surrogate d;
  long chunk;
  unsigned short *X;   // [chunk][32] bf16
  float *pred;         // [chunk][64]
  int *list;           // [list_cap] box-cell indices
  long list_cap;
  int *nfall;          // [1] entries of list
  unsigned long long *counts;  // [2] cells, fallback cells since izem_surr_counts
};

static void surr_free(IzSurr *u) {
  if (!u) return;
  if (u->X) (void)hipFree(u->X);
  if (u->pred) (void)hipFree(u->pred);
  if (u->list) (void)hipFree(u->list);
  if (u->nfall) (void)hipFree(u->nfall);
  if (u->counts) (void)hipFree(u->counts);
  free(u);
}

// ------------------------------------------------------------ kernels
__global__ void k_ckwyr(int n, const double *__restrict__ rho, const double *__restrict__ T,
                        const double *__restrict__ Y, double *__restrict__ wdot) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int kk = c_mech.kk;
  double y[CK_KMAX], w[CK_KMAX];
  for (int k = 0; k < kk; k++) y[k] = Y[(long)t * kk + k];
  d_ckwyr(rho[t], T[t], y, w);
  for (int k = 0; k < kk; k++) wdot[(long)t * kk + k] = w[k];
}

// add per-lane work counters to stats[0..3], one atomic per wave and counter
__device__ inline void chem_stats_add(unsigned long long *stats, unsigned long long a,
                                      unsigned long long b, unsigned long long c,
                                      unsigned long long d) {
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
    c += __shfl_xor(c, off, 64);
    d += __shfl_xor(d, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&stats[0], a);
    atomicAdd(&stats[1], b);
    atomicAdd(&stats[2], c);
    atomicAdd(&stats[3], d);
  }
}

// Where a kernel variant keeps the Nordsieck history.  At one wave per SIMD
// the lane has 512 registers for the kinetics temporaries and the LU
// factors, and the history (7 x N_ doubles, indexed by the current order)
// goes to LDS: 35 KB per 64-lane block, four blocks per CU.  Variants with
// more waves per SIMD keep it in private memory.
#ifndef IZ_ZLDS_MAX_WAVES
#define IZ_ZLDS_MAX_WAVES 1
#endif
#define IZ_ZLDS_DOUBLES(WAVES) ((WAVES) <= IZ_ZLDS_MAX_WAVES ? IZ_ZCOLS * N_ * 64 : 1)

// integrate this lane's cells with the history storage of the variant.  The
// saved Jacobian is the lane's own, kept across its cells and cleared once.
// It stays in private memory (an address the compiler cannot fold keeps it
// from being split into registers): it is written about once per cell and
// read once per step, while 200 of the lane's 512 registers held for it
// meant spills around the kinetics (2^20 flow half steps: 1.26 ms with J in
// registers, 1.07 ms so; 2^18 ignition cells: 31.4 and 28.1 ms).
template <class Kin, int WAVES, class IO>
__device__ IZ_FORCEINLINE void chem_run(double *zs, IO &io, double dt, double rtol, double atol,
                                        int jac_age) {
  double Jm[N_][N_];
  int j0 = 0;
  asm volatile("" : "+v"(j0));
  double (&J)[N_][N_] = *(double (*)[N_][N_])(&Jm[0][0] + j0);
  for (int i = 0; i < N_; i++)
    for (int j = 0; j < N_; j++) J[i][j] = 0.0;
  if constexpr (WAVES <= IZ_ZLDS_MAX_WAVES) {
    ZLds z{zs + threadIdx.x};
    d_bdf_run(Kin(), z, J, io, dt, rtol, atol, jac_age);
  } else {
    ZArr z;
    for (int i = 0; i < IZ_ZCOLS; i++)
      for (int j = 0; j < N_; j++) z.a[i][j] = 0.0;
    d_bdf_run(Kin(), z, J, io, dt, rtol, atol, jac_age);
  }
}

// a lane's work counters
struct ChemCount {
  unsigned long long nst, nfe, nje, nsol;
  __device__ inline void add(const BdfResult &r) {
    nst += r.nst;
    nfe += r.nfe;
    nje += r.nje;
    nsol += r.nsol;
  }
};

// The work queue: a lane takes the next position from a device counter as
// soon as its cell is finished, so lanes stay busy whatever the cells' step
// counts.  Lanes from `lanes` on take none: a small batch is spread over one
// wave per CU (see persistent_grid).
struct PsrQueue {
  int n, lanes;
  double *T;
  const double *rho;
  double *Y;
  int *counter;
  const int *order;
  int *nsteps, *status;
  int cell;
  ChemCount w;
  __device__ inline bool sorted() const { return order != nullptr; }
  __device__ inline bool next(double &r, double *y) {
    if ((int)threadIdx.x >= lanes) return false;
    const int q = atomicAdd(counter, 1);
    if (q >= n) return false;
    cell = order ? order[q] : q;
    r = rho[cell];
    y[0] = T[cell];
#pragma unroll
    for (int k = 0; k < N_ - 1; k++) y[1 + k] = Y[(long)cell * (N_ - 1) + k];
    return true;
  }
  __device__ inline void done(const double *y, const BdfResult &r) {
    T[cell] = y[0];
#pragma unroll
    for (int k = 0; k < N_ - 1; k++) Y[(long)cell * (N_ - 1) + k] = y[1 + k];
    if (nsteps) nsteps[cell] = r.nst;
    if (!r.ok) atomicOr(status, IZ_ST_VODE_FAIL);
    w.add(r);
  }
};

// persistent work-queue kernel over independent cells
template <class Kin, int WAVES>
__global__ void __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(WAVES, WAVES))) k_psr_queue(int n, int lanes, double *__restrict__ T, const double *__restrict__ rho,
                            double *__restrict__ Y, double dt, double rtol, double atol,
                            int jac_age, int *__restrict__ counter,
                            const int *__restrict__ order, int *__restrict__ nsteps,
                            int *__restrict__ status, unsigned long long *__restrict__ stats) {
  __shared__ double zs[IZ_ZLDS_DOUBLES(WAVES)];
  PsrQueue io{n, lanes, T, rho, Y, counter, order, nsteps, status, 0, {0, 0, 0, 0}};
  chem_run<Kin, WAVES>(zs, io, dt, rtol, atol, jac_age);
  chem_stats_add(stats, io.w.nst, io.w.nfe, io.w.nje, io.w.nsol);
}

__device__ inline void atomic_max_posd(double *addr, double val) {
  atomicMax((unsigned long long *)addr, (unsigned long long)__double_as_longlong(val));
}

// the queue over the reacting box of a flow state (i0.., j0.., k0..; ni x nj
// cells per plane): CGS conversion in, T update, DTmax, Y clipping and
// closure out (module_reaction.f90:102-304)
struct FlowQueue {
  IzDims d;
  int i0, j0, k0, ni, nj;
  long n;
  int lanes;
  double T_ref, rho_cgs;
  double *T, *v;
  int *counter;
  const int *order;
  int *status;
  long c;
  double dtmax;
  ChemCount w;
  __device__ inline bool sorted() const { return order != nullptr; }
  __device__ inline bool next(double &r, double *y) {
    if ((int)threadIdx.x >= lanes) return false;
    const long q = atomicAdd(counter, 1);
    if (q >= n) return false;
    const long cell = order ? (long)order[q] : q;
    const int i = i0 + (int)(cell % ni);
    const long p = cell / ni;
    const int j = j0 + (int)(p % nj), k = k0 + (int)(p / nj);
    c = iz_cidx(d, i, j, k);
    const double rho0 = v[c];
    const double rho_i = 1.0 / rho0;
    r = rho0 * rho_cgs;
    y[0] = T[c] * T_ref;
#pragma unroll
    for (int l = 0; l < N_ - 1; l++) y[1 + l] = v[(IZ_NIV + l) * d.nc + c] * rho_i;
    return true;
  }
  __device__ inline void done(const double *y, const BdfResult &r) {
    if (!r.ok) atomicOr(status, IZ_ST_VODE_FAIL);
    w.add(r);
    // the cell's density and start temperature are read again rather than
    // held through the integration
    const double rho0 = v[c];
    dtmax = fmax(dtmax, fabs(y[0] - T[c] * T_ref));
    T[c] = y[0] * (1.0 / T_ref);
    double sumY = 0.0;
#pragma unroll
    for (int l = 0; l < N_ - 2; l++) {
      const double Ya = fmin(fmax(y[1 + l], 0.0), 1.0);
      v[(IZ_NIV + l) * d.nc + c] = rho0 * Ya;
      sumY = sumY + Ya;
    }
    // the last species closes the sum with the unclipped 1 - sum (:293)
    v[(IZ_NIV + N_ - 2) * d.nc + c] = rho0 * (1.0 - sumY);
  }
};

// reaction_dvode on the flow state
template <class Kin, int WAVES>
__global__ void __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(WAVES, WAVES))) k_reaction_queue(IzDims d, int lanes, int i0, int i1, int j0, int j1, int k0, int k1,
                                 const double *__restrict__ dtp, double scale, double time_ref,
                                 double T_ref, double rho_cgs, double rtol, double atol,
                                 int jac_age, double *__restrict__ T, double *__restrict__ v,
                                 int *__restrict__ counter, const int *__restrict__ order,
                                 const int *__restrict__ list_n, double *__restrict__ ts,
                                 int *__restrict__ status,
                                 unsigned long long *__restrict__ stats) {
  __shared__ double zs[IZ_ZLDS_DOUBLES(WAVES)];
  const int ni = i1 - i0 + 1, nj = j1 - j0 + 1, nk = k1 - k0 + 1;
  // list_n: only the first *list_n cells of the list `order` (the
  // surrogate's fallback cells), else every cell of the box
  const long n = list_n ? (long)*list_n : (long)ni * nj * nk;
  const double dt_phys = (scale * (*dtp)) * time_ref;
  FlowQueue io{d, i0, j0, k0, ni, nj, n, lanes, T_ref, rho_cgs, T, v, counter, order, status,
               0, 0.0, {0, 0, 0, 0}};
  chem_run<Kin, WAVES>(zs, io, dt_phys, rtol, atol, jac_age);
  double dtmax = io.dtmax;
  for (int off = 32; off > 0; off >>= 1) dtmax = fmax(dtmax, __shfl_xor(dtmax, off, 64));
  if ((threadIdx.x & 63) == 0) atomic_max_posd(&ts[5], dtmax);
  chem_stats_add(stats, io.w.nst, io.w.nfe, io.w.nje, io.w.nsol);
}

__global__ void k_stats_zero(unsigned long long *stats) {
  if (threadIdx.x < 4) stats[threadIdx.x] = 0ull;
}

__global__ void k_chem_prep(int *counter, double *ts, int zero_dtmax) {
  *counter = 0;
  if (zero_dtmax) ts[5] = 0.0;
}

// ------------------------------------------------------------------ host
// the straight-line kinetics are used only when they agree with the loaded
// tables: both are evaluated on the device at a few states
__global__ void k_gen_check(int *ok) {
  const double Ts[3] = {700.0, 1300.0, 2600.0};
  int good = 1;
  for (int q = 0; q < 3; q++) {
    double y[CK_NEQ], f1[CK_NEQ], f2[CK_NEQ];
    y[0] = Ts[q];
    for (int k = 0; k < CK_NEQ - 1; k++) y[1 + k] = (k + 1.0) / 45.0;
    KinGen().rhs(3e-4, y, f1);
    KinTables().rhs(3e-4, y, f2);
    for (int i = 0; i < CK_NEQ; i++)
      if (!(fabs(f1[i] - f2[i]) <= 1e-9 * fabs(f2[i]) + 1e-20)) good = 0;
  }
  *ok = good;
}

// Scratch of izem_psr_batch_noalloc, one copy per GPU for the life of the
// process: the work-queue head, the stiffness order's bin counts, then the
// cells' bins and the queue permutation of up to IZEM_NOALLOC_MAX_CELLS
// cells: 4 (2 IZEM_NOALLOC_MAX_CELLS + 576) bytes, about 8 MB.  Host code
// uses the address noalloc_scratch returns, never the symbol itself.
#define IZ_NOALLOC_HIST 64
#define IZ_NOALLOC_BIN (IZ_NOALLOC_HIST + IZ_ORDER_BINS)
#define IZ_NOALLOC_PERM (IZ_NOALLOC_BIN + IZEM_NOALLOC_MAX_CELLS)
static __device__ __align__(256) int scratch[IZ_NOALLOC_PERM + IZEM_NOALLOC_MAX_CELLS];

#define IZ_MAX_DEVICES 64
static int *g_scratch[IZ_MAX_DEVICES];

// device address of the current GPU's scratch, looked up once per device
static int noalloc_scratch(int **base) {
  int dev = 0;
  IZ_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= IZ_MAX_DEVICES) return IZEM_E_STATE;
  if (!g_scratch[dev]) {
    void *p = nullptr;
    IZ_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[dev] = (int *)p;
  }
  *base = g_scratch[dev];
  return IZEM_OK;
}

void iz_chem_destroy(izem_ctx *ctx) {
  if (!ctx || !ctx->chem) return;
  if (ctx->chem->counter) (void)hipFree(ctx->chem->counter);
  if (ctx->chem->stats) (void)hipFree(ctx->chem->stats);
  if (ctx->chem->order_hist) (void)hipFree(ctx->chem->order_hist);
  if (ctx->chem->order_bin) (void)hipFree(ctx->chem->order_bin);
  if (ctx->chem->order_perm) (void)hipFree(ctx->chem->order_perm);
  surr_free(ctx->chem->surr);
  free(ctx->chem);
  ctx->chem = nullptr;
}

// Setup self-check of the straight-line kinetics' compiled integrator: 64
// ignition cells (stoichiometric H2/air at 1 atm, 1000..1630 K, over
// 1e-6 s) integrated by the one-wave kernel with both straight-line forms
// and with the table-driven kinetics.  They differ in round-off and in the
// iteration matrix only, so end
// temperatures agree to 1e-6 relative and the step totals to 3 %; a build
// of the straight-line kernel that departs from its source (as some builds
// of its heavily spilling variants did) fails this and the context does
// without that form.  ok: bit f - 1 set where form f agrees.  The work
// counters and the status word are not touched.
static int gen_bdf_check(izem_ctx *ctx, const IzMech &m, int &ok) {
  constexpr int n = 64, nsp = CK_NEQ - 1;
  const double dt = 1.0e-6;
  double T[3][n], rho[n], Y[3][n * nsp];
  int nst[3][n];
  for (int c = 0; c < n; c++) {
    double y[nsp] = {0.0, 0.0283, 0.0, 0.2264, 0.0, 0.0, 0.0, 0.0, 0.0};
    y[0] = 1.0e-6 * (1 + c % 4);           // a trace of H atoms
    y[4] = 1.0e-6 * (1 + (c / 4) % 4);     // and of OH
    double s = 0.0;
    for (int k = 0; k < nsp - 1; k++) s += y[k];
    y[nsp - 1] = 1.0 - s;                  // N2 closes the sum
    double wi = 0.0;
    for (int k = 0; k < nsp; k++) wi += y[k] / m.wt[k];
    T[0][c] = T[1][c] = T[2][c] = 1000.0 + 10.0 * c;
    rho[c] = 1.01325e6 / (8.314510e7 * T[0][c] * wi);
    for (int k = 0; k < nsp; k++) Y[0][c * nsp + k] = Y[1][c * nsp + k] = Y[2][c * nsp + k] = y[k];
  }
  double *dT = nullptr, *dr = nullptr, *dY = nullptr;
  int *dn = nullptr, *dst = nullptr;
  unsigned long long *dstats = nullptr;  // the check's own work counters
  int rc = IZEM_OK;
  IzChem *ch = ctx->chem;
  if (hipMalloc(&dT, sizeof T[0]) != hipSuccess || hipMalloc(&dr, sizeof rho) != hipSuccess ||
      hipMalloc(&dY, sizeof Y[0]) != hipSuccess || hipMalloc(&dn, sizeof nst[0]) != hipSuccess ||
      hipMalloc(&dst, sizeof(int)) != hipSuccess ||
      hipMalloc(&dstats, 4 * sizeof(unsigned long long)) != hipSuccess) {
    rc = IZEM_E_NOMEM;
  } else {
    hipLaunchKernelGGL(k_stats_zero, dim3(1), dim3(64), 0, ctx->stream, dstats);
    int zero = 0;
    for (int v = 0; v < 3 && rc == IZEM_OK; v++) {
      if (hipMemcpyAsync(dT, T[v], sizeof T[0], hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
          hipMemcpyAsync(dr, rho, sizeof rho, hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
          hipMemcpyAsync(dY, Y[v], sizeof Y[0], hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
          hipMemcpyAsync(dst, &zero, sizeof zero, hipMemcpyHostToDevice, ctx->stream) != hipSuccess) {
        rc = IZEM_E_HIP;
        break;
      }
      hipLaunchKernelGGL(k_chem_prep, dim3(1), dim3(1), 0, ctx->stream, ch->counter, ctx->ts, 0);
#define IZ_CHECK_PSR(K)                                                                         \
  hipLaunchKernelGGL((k_psr_queue<K, 1>), dim3(1), dim3(64), 0, ctx->stream, n, 64, dT, dr, dY, dt, \
                     ch->rtol, ch->atol, ch->jac_age, ch->counter, nullptr, dn, dst, dstats)
      if (v == 0) IZ_CHECK_PSR(KinTables);
      else if (v == 1) IZ_CHECK_PSR(KinGen);
      else IZ_CHECK_PSR(KinGenAJ);
#undef IZ_CHECK_PSR
      if (hipGetLastError() != hipSuccess ||
          hipMemcpyAsync(T[v], dT, sizeof T[0], hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
          hipMemcpyAsync(nst[v], dn, sizeof nst[0], hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
          hipStreamSynchronize(ctx->stream) != hipSuccess)
        rc = IZEM_E_HIP;
    }
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) rc = IZEM_E_HIP;
  }
  if (dstats) (void)hipFree(dstats);
  if (dT) (void)hipFree(dT);
  if (dr) (void)hipFree(dr);
  if (dY) (void)hipFree(dY);
  if (dn) (void)hipFree(dn);
  if (dst) (void)hipFree(dst);
  if (rc != IZEM_OK) return rc;
  ok = 0;
  for (int v = 1; v < 3; v++)
    if (iz_forms_agree(n, T[0], nst[0], T[v], nst[v])) ok |= 1 << (v - 1);
  return IZEM_OK;
}

extern "C" int izem_chem_setup(izem_ctx *ctx, const double *mf, long nmech, double rtol,
                               double atol, int trim) {
  if (!ctx || !mf || rtol <= 0 || atol <= 0) return IZEM_E_ARG;
  IzMech m;
  if (!iz_mech_from_flat(mf, nmech, CK_NEQ - 1, m)) return IZEM_E_ARG;
  IzBdf bt;
  iz_bdf_tables(bt);
  IZ_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_mech), &m, sizeof m));
  IZ_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_bdf), &bt, sizeof bt));
  if (!ctx->chem) {
    ctx->chem = (IzChem *)calloc(1, sizeof(IzChem));
    if (!ctx->chem) return IZEM_E_NOMEM;
    if (hipMalloc(&ctx->chem->counter, sizeof(int)) != hipSuccess ||
        hipMalloc(&ctx->chem->stats, 4 * sizeof(unsigned long long)) != hipSuccess ||
        hipMalloc(&ctx->chem->order_hist, IZ_ORDER_BINS * sizeof(int)) != hipSuccess) {
      iz_chem_destroy(ctx);  // frees what was allocated, ctx->chem = nullptr
      return IZEM_E_NOMEM;
    }
    ctx->chem->order = 0;
    hipLaunchKernelGGL(k_stats_zero, dim3(1), dim3(64), 0, ctx->stream, ctx->chem->stats);
    // defaults measured on MI355X (2^18 cells at dt = 1e-6 s and 2^20 cells
    // of a reacting HIT half step): one wave per SIMD with the whole
    // register file, the factors in registers and the history in LDS
    ctx->chem->waves = 1;
    ctx->chem->blocks_per_cu = 4;
    ctx->chem->jac_age = 50;  // DVODE MSBJ
  }
  int same = 0;
  if (m.kk == GEN_KK && m.ii == GEN_II) {
    hipLaunchKernelGGL(k_gen_check, dim3(1), dim3(1), 0, ctx->stream, ctx->chem->counter);
    IZ_CHECK(hipMemcpyAsync(&same, ctx->chem->counter, sizeof(int), hipMemcpyDeviceToHost,
                            ctx->stream));
    IZ_CHECK(hipStreamSynchronize(ctx->stream));
  }
  {
    // locate this GPU's scratch of izem_psr_batch_noalloc at set-up
    int *base = nullptr;
    const int rs = noalloc_scratch(&base);
    if (rs != IZEM_OK) return rs;
  }
  ctx->chem->rtol = rtol;
  ctx->chem->atol = atol;
  ctx->chem->trim = trim;
  ctx->chem->generated = 0;
  if (same) {
    int rc = gen_bdf_check(ctx, m, ctx->chem->generated);
    if (rc != IZEM_OK) return rc;
  }
  // the closed-form Jacobian is the faster straight-line form on short and
  // long substeps alike (2^20 flow half steps: 1.07 against 1.38 ms; 2^18
  // ignition cells: 28 against 34 ms)
  ctx->chem->use_gen = iz_chem_form(ctx->chem->generated, 1, -1);
  return IZEM_OK;
}

// parameters chosen by phd_amd.autotune: register budget, persistent blocks
// per CU, Jacobian reuse age, kinetics form (0 tables, 1 straight-line,
// 2 straight-line with the closed-form Jacobian, -1 that form when it matches
// the loaded mechanism and the budget).
// The straight-line kinetics run at one wave per SIMD only: builds of them
// at two and four waves per SIMD (history in private memory, several KB of
// spills per lane) were seen to take other steps than a host build of the
// same source, with the variant affected changing from one build to the
// next, while the one-wave build follows it.
extern "C" int izem_chem_tune(izem_ctx *ctx, int waves, int blocks_per_cu, int jac_age,
                              int kinetics) {
  if (!ctx || !ctx->chem || !(waves == 1 || waves == 2 || waves == 4) || blocks_per_cu < 1 ||
      blocks_per_cu > 64 || jac_age < 1 || kinetics < -1 || kinetics > 2)
    return IZEM_E_ARG;
  const int form = iz_chem_form(ctx->chem->generated, waves, kinetics);
  if (form < 0) return IZEM_E_ARG;
  ctx->chem->use_gen = form;
  ctx->chem->waves = waves;
  ctx->chem->blocks_per_cu = blocks_per_cu;
  ctx->chem->jac_age = jac_age;
  return IZEM_OK;
}

// ---------------------------------------------------- stiffness order
// Lanes take cells one after the other, so what is left of a wave's idle
// time is the end of the launch, where lanes with long last cells run on.
// izem_psr_batch can hand cells out in decreasing order of a stiffness key, the largest
// diagonal entry of the species block of the reactor Jacobian (the fastest
// chemical rate), so the stiffest come first and neighbouring lanes have
// cells of like step counts.  Each cell is still integrated on its own; only
// the order in which lanes take cells changes.  Counting sort in three passes:
// key and bin counts, exclusive scan, scatter with block-aggregated atomics.
__global__ void k_order_zero(int *__restrict__ hist) {
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x) hist[i] = 0;
}

// queue slot of a cell of density rho [g/cm3] and state y = (T [K], Y_k):
// decreasing key -> increasing slot; NaN keys go last, infinite first
__device__ inline int order_slot(double rho, const double *y) {
  double f0[N_], yl[N_], f[N_];
  d_reactor_rhs(rho, y, f0);
  double s = 0.0;
  for (int j = 1; j < N_; j++) {
    for (int k = 0; k < N_; k++) yl[k] = y[k];
    const double dy = 1.4901161193847656e-08 * fmax(fabs(y[j]), 1.0e-6);
    yl[j] = y[j] + dy;
    d_reactor_rhs(rho, yl, f);
    s = fmax(s, fabs((f[j] - f0[j]) / dy));
  }
  const double l = log2(s) * 8.0;
  const int b = (l >= 1.0) ? (l < IZ_ORDER_BINS - 1 ? (int)l : IZ_ORDER_BINS - 1) : 0;
  return IZ_ORDER_BINS - 1 - b;
}

__global__ void __launch_bounds__(256) k_order_key(int n, const double *__restrict__ T,
                                                   const double *__restrict__ rho,
                                                   const double *__restrict__ Y,
                                                   int *__restrict__ bin,
                                                   int *__restrict__ hist) {
  __shared__ int h[IZ_ORDER_BINS];
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x) h[i] = 0;
  __syncthreads();
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) {
    double y[N_];
    y[0] = T[c];
    for (int k = 0; k < N_ - 1; k++) y[1 + k] = Y[(long)c * (N_ - 1) + k];
    const int slot = order_slot(rho[c], y);
    bin[c] = slot;
    atomicAdd(&h[slot], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// the same key on the cells of the reacting box of the flow state, in the
// queue numbering of k_reaction_queue (i fastest) and its unit conversion
__global__ void __launch_bounds__(256) k_order_key_flow(IzDims d, int i0, int j0, int k0, int ni,
                                                        int nj, int n, double T_ref,
                                                        double rho_cgs,
                                                        const double *__restrict__ T,
                                                        const double *__restrict__ v,
                                                        int *__restrict__ bin,
                                                        int *__restrict__ hist) {
  __shared__ int h[IZ_ORDER_BINS];
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x) h[i] = 0;
  __syncthreads();
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) {
    const int i = i0 + q % ni;
    const int r = q / ni;
    const long c = iz_cidx(d, i, j0 + r % nj, k0 + r / nj);
    const double rho0 = v[c];
    double y[N_];
    y[0] = T[c] * T_ref;
    for (int l = 0; l < N_ - 1; l++) y[1 + l] = v[(IZ_NIV + l) * d.nc + c] / rho0;
    const int slot = order_slot(rho0 * rho_cgs, y);
    bin[q] = slot;
    atomicAdd(&h[slot], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// counts -> exclusive offsets, in place (one 64-lane block)
__global__ void k_order_scan(int *__restrict__ hist) {
  __shared__ int part[64];
  constexpr int per = IZ_ORDER_BINS / 64;
  const int t = threadIdx.x;
  int loc[per], sum = 0;
  for (int i = 0; i < per; i++) {
    loc[i] = sum;
    sum += hist[t * per + i];
  }
  part[t] = sum;
  __syncthreads();
  if (t == 0) {
    int run = 0;
    for (int i = 0; i < 64; i++) {
      const int v = part[i];
      part[i] = run;
      run += v;
    }
  }
  __syncthreads();
  for (int i = 0; i < per; i++) hist[t * per + i] = part[t] + loc[i];
}

__global__ void __launch_bounds__(256) k_order_scatter(int n, const int *__restrict__ bin,
                                                       int *__restrict__ off,
                                                       int *__restrict__ perm) {
  __shared__ int h[IZ_ORDER_BINS];
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x) h[i] = 0;
  __syncthreads();
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  int slot = 0, rank = 0;
  if (c < n) {
    slot = bin[c];
    rank = atomicAdd(&h[slot], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < IZ_ORDER_BINS; i += blockDim.x)
    if (h[i]) h[i] = atomicAdd(&off[i], h[i]);
  __syncthreads();
  if (c < n) perm[h[slot] + rank] = c;
}

// queue permutation of n cells: order_begin sizes the buffers and clears
// the bin counts (IZEM_E_NOMEM if the buffers cannot grow), a key kernel
// writes the bins and counts, order_end scans and scatters
static int order_begin(izem_ctx *ctx, int n) {
  IzChem *ch = ctx->chem;
  if (n > ch->order_cap) {
    IZ_CHECK(hipStreamSynchronize(ctx->stream));
    if (ch->order_bin) (void)hipFree(ch->order_bin);
    if (ch->order_perm) (void)hipFree(ch->order_perm);
    ch->order_bin = ch->order_perm = nullptr;
    ch->order_cap = 0;
    if (hipMalloc(&ch->order_bin, (size_t)n * sizeof(int)) != hipSuccess ||
        hipMalloc(&ch->order_perm, (size_t)n * sizeof(int)) != hipSuccess)
      return IZEM_E_NOMEM;
    ch->order_cap = n;
  }
  hipLaunchKernelGGL(k_order_zero, dim3(1), dim3(256), 0, ctx->stream, ch->order_hist);
  return IZEM_OK;
}

static int order_end(izem_ctx *ctx, int n, const int *bin, int *hist, int *perm) {
  const int nb = (n + 255) / 256;
  hipLaunchKernelGGL(k_order_scan, dim3(1), dim3(64), 0, ctx->stream, hist);
  hipLaunchKernelGGL(k_order_scatter, dim3(nb), dim3(256), 0, ctx->stream, n, bin, hist, perm);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// the chemistry settings a captured step bakes into its kernel arguments;
// IZEM_E_STATE with the stiffness order on (its buffers may grow, which
// allocates and synchronises)
int iz_chem_signature(izem_ctx *ctx, double sig[IZ_CHEM_SIG]) {
  IzChem *ch = ctx->chem;
  if (!ch) return IZEM_E_STATE;
  if (ch->order) return IZEM_E_STATE;
  const double s[IZ_CHEM_SIG] = {(double)ch->use_gen, (double)ch->waves,
                                 (double)ch->blocks_per_cu, (double)ch->jac_age, ch->rtol,
                                 ch->atol, (double)ch->trim, (double)ch->sel_gen};
  for (int i = 0; i < IZ_CHEM_SIG; i++) sig[i] = s[i];
  return IZEM_OK;
}

extern "C" int izem_chem_order(izem_ctx *ctx, int on) {
  if (!ctx || !ctx->chem || on < 0 || on > 1) return IZEM_E_ARG;
  ctx->chem->order = on;
  return IZEM_OK;
}

extern "C" int izem_chem_order_read(izem_ctx *ctx, long cap, long *n, int *perm, int *bin) {
  if (!ctx || !ctx->chem || !n || cap < 0) return IZEM_E_ARG;
  IzChem *ch = ctx->chem;
  IZ_CHECK(hipStreamSynchronize(ctx->stream));
  *n = ch->order_n;
  if (ch->order_n == 0) return IZEM_OK;
  if (ch->order_n > cap || !perm || !bin) return IZEM_E_ARG;
  IZ_CHECK(hipMemcpy(perm, ch->order_perm, ch->order_n * sizeof(int), hipMemcpyDeviceToHost));
  IZ_CHECK(hipMemcpy(bin, ch->order_bin, ch->order_n * sizeof(int), hipMemcpyDeviceToHost));
  return IZEM_OK;
}

// blocks of a persistent launch over n cells, and the lanes of each that take
// cells.  Up to one full wave per CU (64 cells per CU, whatever the tuned
// blocks per CU) the cells are spread over all the CUs, one wave on each:
// a wave of few cells seldom runs the branches (Jacobian, pivoting, third
// corrector iteration) that only some cells need, and the launch lasts as
// long as its slowest cell's chain of steps (1000 ignition cells: 10.9 ms
// as 16 full waves, 8.8 ms as 250 waves of four).  Beyond that the waves
// are full (one wave per SIMD already shares its CU's caches with three
// others: 14400 cells of three steps take 0.075 ms as 225 full waves, 0.10
// ms as 960 waves of 15).
static int persistent_grid(izem_ctx *ctx, long n, int *lanes) {
  const long ncu = ctx->ncu;
  *lanes = 64;
  if (n <= 64 * ncu) {
    const long g = n < ncu ? n : ncu;
    *lanes = (int)((n + g - 1) / (g < 1 ? 1 : g));
    if (*lanes < 1) *lanes = 1;
    return (int)(g < 1 ? 1 : g);
  }
  long g = ncu * ctx->chem->blocks_per_cu;
  const long maxg = (n + 63) / 64;
  if (g > maxg) g = maxg;
  return (int)g;
}

extern "C" int izem_ckwyr(izem_ctx *ctx, int n, const double *rho, const double *T,
                          const double *Y, double *wdot) {
  if (!ctx || !ctx->chem || n < 0 || !rho || !T || !Y || !wdot) return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  hipLaunchKernelGGL(k_ckwyr, dim3(iz_blocks(n, 128)), dim3(128), 0, ctx->stream, n, rho, T, Y,
                     wdot);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// reset the queue head and run the persistent reactor kernel of the tuned
// variant over n cells (queue position q takes cell order[q], or q)
static void psr_launch(izem_ctx *ctx, dim3 grid, int lanes, int n, double *T, const double *rho, double *Y,
                       double dt, int *counter, const int *order, int *nsteps) {
  IzChem *ch = ctx->chem;
  hipLaunchKernelGGL(k_chem_prep, dim3(1), dim3(1), 0, ctx->stream, counter, ctx->ts, 0);
#define IZ_PSR(K, W)                                                                            \
  hipLaunchKernelGGL((k_psr_queue<K, W>), grid, dim3(64), 0, ctx->stream, n, lanes, T, rho, Y, dt, \
                     ch->rtol, ch->atol, ch->jac_age, counter, order, nsteps, ctx->status,      \
                     ch->stats)
  if (ch->use_gen == 2) {
    IZ_PSR(KinGenAJ, 1);
  } else if (ch->use_gen) {
    IZ_PSR(KinGen, 1);
  } else {
    if (ch->waves == 1) IZ_PSR(KinTables, 1);
    else if (ch->waves == 2) IZ_PSR(KinTables, 2);
    else IZ_PSR(KinTables, 4);
  }
#undef IZ_PSR
}

extern "C" int izem_psr_batch(izem_ctx *ctx, int n, double *T, const double *rho, double *Y,
                              double dt, int *nsteps) {
  if (!ctx || !ctx->chem || n < 0 || !T || !rho || !Y || !(dt > 0)) return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  IzChem *ch = ctx->chem;
  int pk = iz_prof_begin(ctx, IZP_CHEM);
  int lanes;
  dim3 grid(persistent_grid(ctx, n, &lanes));
  const int *order = nullptr;
  // with no more cells than resident lanes each lane takes one cell and the
  // batch lasts as long as its stiffest cell in any order
  if (ch->order && (long)n > 64L * grid.x) {
    int rc = order_begin(ctx, n);
    if (rc == IZEM_OK) {
      hipLaunchKernelGGL(k_order_key, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, T, rho,
                         Y, ch->order_bin, ch->order_hist);
      rc = order_end(ctx, n, ch->order_bin, ch->order_hist, ch->order_perm);
    }
    if (rc != IZEM_OK) {
      iz_prof_end(ctx, pk);
      return rc;
    }
    order = ch->order_perm;
  }
  ch->order_n = order ? n : 0;
  psr_launch(ctx, grid, lanes, n, T, rho, Y, dt, ch->counter, order, nsteps);
  iz_prof_end(ctx, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_psr_batch_noalloc(izem_ctx *ctx, int n, double *T, const double *rho,
                                      double *Y, double dt, int *nsteps) {
  if (!ctx || !ctx->chem || n < 0 || !T || !rho || !Y || !(dt > 0)) return IZEM_E_ARG;
  if (n > IZEM_NOALLOC_MAX_CELLS) return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  int *base = nullptr;
  const int rs = noalloc_scratch(&base);
  if (rs != IZEM_OK) return rs;
  int *counter = base, *hist = base + IZ_NOALLOC_HIST, *bin = base + IZ_NOALLOC_BIN,
      *perm = base + IZ_NOALLOC_PERM;
  IzChem *ch = ctx->chem;
  int pk = iz_prof_begin(ctx, IZP_CHEM);
  int lanes;
  dim3 grid(persistent_grid(ctx, n, &lanes));
  const int *order = nullptr;
  if (ch->order && (long)n > 64L * grid.x) {
    hipLaunchKernelGGL(k_order_zero, dim3(1), dim3(256), 0, ctx->stream, hist);
    hipLaunchKernelGGL(k_order_key, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, T, rho,
                       Y, bin, hist);
    const int rc = order_end(ctx, n, bin, hist, perm);
    if (rc != IZEM_OK) {
      iz_prof_end(ctx, pk);
      return rc;
    }
    order = perm;
  }
  psr_launch(ctx, grid, lanes, n, T, rho, Y, dt, counter, order, nsteps);
  iz_prof_end(ctx, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// reacting box: module_reaction.f90:138-150 (trimmed by ng+1 at the global
// faces unless trim == 0); in 2-D the z range is the whole box
struct IzBox {
  int i0, i1, j0, j1, k0, k1;
  long n;
};
static IzBox react_box(const izem_ctx *ctx) {
  const IzDims &d = ctx->d;
  IzBox b{0, d.nx - 1, 0, d.ny - 1, 0, d.nz - 1, 0};
  if (ctx->chem->trim) {
    b.i0 = d.ng; b.i1 = d.nx - d.ng - 2;
    b.j0 = d.ng; b.j1 = d.ny - d.ng - 2;
    if (d.ndim == 3) {
      // fz = min(ey, ntz-ng-1): the reference bounds z by the y extent
      b.k0 = d.ng;
      b.k1 = d.nz - d.ng - 2;
      if (b.k1 > d.ny - 1) b.k1 = d.ny - 1;
    }
  }
  if (b.i1 < b.i0 || b.j1 < b.j0 || b.k1 < b.k0) return b;
  b.n = (long)(b.i1 - b.i0 + 1) * (b.j1 - b.j0 + 1) * (b.k1 - b.k0 + 1);
  return b;
}

// the persistent reactor kernel of the tuned variant over the box's cells
// (queue position q takes box cell order[q], or q; with list_n the first
// *list_n entries of order only)
static void reaction_queue(izem_ctx *ctx, const IzBox &b, dim3 grid, int lanes, const double *dt,
                           double scale, double *T, double *v, const int *order,
                           const int *list_n) {
  IzChem *ch = ctx->chem;
  const double rho_cgs = ctx->o.rho_ref * 1.0e-3;
#define IZ_RQ(K, W)                                                                             \
  hipLaunchKernelGGL((k_reaction_queue<K, W>), grid, dim3(64), 0, ctx->stream, ctx->d, lanes, b.i0, \
                     b.i1, b.j0, b.j1, b.k0, b.k1, dt, scale, ctx->o.time_ref, ctx->o.T_ref,    \
                     rho_cgs, ch->rtol, ch->atol, ch->jac_age, T, v, ch->counter, order, list_n, \
                     ctx->ts, ctx->status, ch->stats)
  if (ch->use_gen == 2) {
    IZ_RQ(KinGenAJ, 1);
  } else if (ch->use_gen) {
    IZ_RQ(KinGen, 1);
  } else {
    if (ch->waves == 1) IZ_RQ(KinTables, 1);
    else if (ch->waves == 2) IZ_RQ(KinTables, 2);
    else IZ_RQ(KinTables, 4);
  }
#undef IZ_RQ
}

// the tail of reaction_selec (module_reaction.f90:79-83): W_i, cp, ha
// from the new T and Y, ghost fill, ghost-slab primitives
static int reaction_tail(izem_ctx *ctx, const double *dt, double scale, double *T, double *W_i,
                         double *cp, double *ha, double *v) {
  int r = iz_upd_prim_woT(ctx, 0, v, T, W_i, cp, ha);
  if (r) return r;
  return iz_fill_ghost_newton(ctx, T, W_i, cp, ha, v, dt, scale);
}

extern "C" int izem_reaction_dvode(izem_ctx *ctx, const double *dt, double scale, double *T,
                                   double *W_i, double *cp, double *ha, double *v) {
  if (!ctx || !ctx->chem || !dt || !T || !W_i || !cp || !ha || !v) return IZEM_E_ARG;
  const IzDims &d = ctx->d;
  IzChem *ch = ctx->chem;
  const IzBox b = react_box(ctx);
  const long n = b.n;
  hipLaunchKernelGGL(k_chem_prep, dim3(1), dim3(1), 0, ctx->stream, ch->counter, ctx->ts, 1);
  if (n > 0) {
    double rho_cgs = ctx->o.rho_ref * 1.0e-3;
    int pk = iz_prof_begin(ctx, IZP_CHEM);
    int lanes;
    dim3 grid(persistent_grid(ctx, n, &lanes));
    const int *order = nullptr;
    if (ch->order && n <= INT_MAX && n > 64L * grid.x) {
      const int ni = b.i1 - b.i0 + 1, nj = b.j1 - b.j0 + 1;
      int rc = order_begin(ctx, (int)n);
      if (rc == IZEM_OK) {
        hipLaunchKernelGGL(k_order_key_flow, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                           ctx->stream, d, b.i0, b.j0, b.k0, ni, nj, (int)n, ctx->o.T_ref,
                           rho_cgs, T, v, ch->order_bin, ch->order_hist);
        rc = order_end(ctx, (int)n, ch->order_bin, ch->order_hist, ch->order_perm);
      }
      if (rc != IZEM_OK) {
        iz_prof_end(ctx, pk);
        return rc;
      }
      order = ch->order_perm;
    }
    ch->order_n = order ? n : 0;
    reaction_queue(ctx, b, grid, lanes, dt, scale, T, v, order, nullptr);
    iz_prof_end(ctx, pk);
    IZ_CHECK(hipGetLastError());
  }
  return reaction_tail(ctx, dt, scale, T, W_i, cp, ha, v);
}

// work counters of the chemistry integrations since the previous call
// (BDF steps, RHS evaluations, Jacobians, LU solves); synchronises the
// context stream and clears the counters
extern "C" int izem_chem_stats(izem_ctx *ctx, unsigned long long *out) {
  if (!ctx || !ctx->chem || !out) return IZEM_E_ARG;
  IZ_CHECK(hipMemcpyAsync(out, ctx->chem->stats, 4 * sizeof(unsigned long long),
                          hipMemcpyDeviceToHost, ctx->stream));
  hipLaunchKernelGGL(k_stats_zero, dim3(1), dim3(64), 0, ctx->stream, ctx->chem->stats);
  IZ_CHECK(hipStreamSynchronize(ctx->stream));
  return IZEM_OK;
}

// ===================================================================
// Chemistry surrogate: features, conservation projection, energy-
// consistent temperature, error indicator and the VODE fallback.  No
// counterpart in the reference; the fallback is izem_psr_batch.
// ===================================================================
#define IZ_SURR_NF 12   // features: ln p, T, Y_k (9), ln dt
#define IZ_SURR_XLD 32  // padded feature row (BF16)
#define IZ_SURR_NO 10   // outputs: dT, dY_k (9)

__device__ inline unsigned short surr_f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

// mixture internal energy [erg/g] and c_v [erg/(g K)] from the mechanism's
// NASA-7 tables (CKUMS/CKCVBS forms, chemkin/vode.f:64, 228)
__device__ inline double d_u_mix(double T, const double *Y, double &cv) {
  const double ru = 8.314510e7;  // erg/(mol K), as CKINIT
  double u = 0.0;
  cv = 0.0;
  for (int k = 0; k < CK_NEQ - 1; k++) {
    const double *a = IZ_CMECH.a[k][(T > IZ_CMECH.tmid[k]) ? 1 : 0];
    const double w = IZ_CMECH.wt[k];
    const double h = ru * T * (a[0] + a[1] * T / 2.0 + a[2] * T * T / 3.0 +
                               a[3] * T * T * T / 4.0 + a[4] * T * T * T * T / 5.0 + a[5] / T) / w;
    const double cp = ru * (a[0] + a[1] * T + a[2] * T * T + a[3] * T * T * T +
                            a[4] * T * T * T * T) / w;
    u += Y[k] * (h - ru * T / w);
    cv += Y[k] * (cp - ru / w);
  }
  return u;
}

// one normalised bf16 feature row (ln p, T, Y_k, ln dt) of a cell in
// CHEMKIN units (K, g/cm^3)
__device__ inline void surr_row(double T, double rho, const double *y, double lndt,
                                const float *__restrict__ mean, const float *__restrict__ istd,
                                unsigned short *__restrict__ row) {
  double wi = 0.0;
  float f[IZ_SURR_NF];
  for (int k = 0; k < CK_NEQ - 1; k++) {
    wi += y[k] / IZ_CMECH.wt[k];
    f[2 + k] = (float)y[k];
  }
  const double p = rho * 8.314510e7 * T * wi;  // dyn/cm^2
  f[0] = (float)log(p);
  f[1] = (float)T;
  f[11] = (float)lndt;
  for (int j = 0; j < IZ_SURR_NF; j++) row[j] = surr_f2bf((f[j] - mean[j]) * istd[j]);
  for (int j = IZ_SURR_NF; j < IZ_SURR_XLD; j++) row[j] = 0;
}

__global__ void k_surr_features(int n, const double *__restrict__ T, const double *__restrict__ rho,
                                const double *__restrict__ Y, double lndt,
                                const float *__restrict__ mean, const float *__restrict__ istd,
                                unsigned short *__restrict__ X) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  double y[CK_NEQ - 1];
  for (int k = 0; k < CK_NEQ - 1; k++) y[k] = Y[(long)c * (CK_NEQ - 1) + k];
  surr_row(T[c], rho[c], y, lndt, mean, istd, X + (long)c * IZ_SURR_XLD);
}

// the network's substep for one cell: decode the scaled outputs (dT, dY_k)
// of pred, project dY onto element (hence mass) conservation, and run the
// error indicator.  Returns 1 when the cell must fall back to the BDF path:
// a normalised feature beyond feat_lim (outside the training range), a
// projected mass fraction below -1e-7, or the temperature that keeps the
// mixture internal energy of the constant-volume reactor with the projected
// Y (Newton on u(T, Y1) = u(T0, Y0)) differing from T0 + dT by more than
// tol_T, or |dT| > dT_max.  y1 and dT receive the substep, Te that energy
// temperature.
__device__ inline int surr_decide(const double *y0, double T0, const float *__restrict__ pr,
                                  const float *__restrict__ omean,
                                  const float *__restrict__ ostd, const float *__restrict__ oc,
                                  const double *__restrict__ proj,
                                  const unsigned short *__restrict__ xrow, float feat_lim,
                                  double tol_T, double dT_max, double *y1, double &dT,
                                  double &Te) {
  const int K = CK_NEQ - 1;
  double dy[CK_NEQ - 1];
  // outputs are standardised asinh(change / oc): the transform resolves
  // small and large changes with the same relative accuracy
  dT = oc[0] * sinh((double)(pr[0] * ostd[0] + omean[0]));
  for (int k = 0; k < K; k++)
    dy[k] = oc[1 + k] * sinh((double)(pr[1 + k] * ostd[1 + k] + omean[1 + k]));
  int bad = 0;
  for (int j = 0; j < IZ_SURR_NF; j++) {
    const float x = __uint_as_float(((unsigned)xrow[j]) << 16);
    if (!(fabsf(x) <= feat_lim)) bad = 1;
  }
  double ymin = 1.0;
  for (int i = 0; i < K; i++) {
    double s = 0.0;
    for (int k = 0; k < K; k++) s += proj[i * K + k] * dy[k];
    y1[i] = y0[i] + s;
    ymin = fmin(ymin, y1[i]);
  }
  // a projected mass fraction below -1e-7 rejects the cell; smaller
  // undershoots (absent radicals) are kept, which keeps the element
  // masses exact
  if (!(ymin >= -1.0e-7)) bad = 1;
  double cv;
  const double u0 = d_u_mix(T0, y0, cv);
  // converged to 1e-12 relative (about 1e-9 K), far below the smallest
  // tol_T a calibration on slowly reacting cells picks
  Te = T0 + dT;
  for (int it = 0; it < 10; it++) {
    const double u = d_u_mix(Te, y1, cv);
    const double d = (u - u0) / cv;
    Te -= d;
    if (fabs(d) < 1.0e-12 * Te) break;
  }
  if (!(fabs(Te - (T0 + dT)) <= tol_T) || !(fabs(dT) <= dT_max) || !(Te > 0.0)) bad = 1;
  return bad;
}

// accept or reject the network's substep for each of n packed cells; on
// acceptance Y += proj.dY and T += dT.  flag: 0 accepted, 1 fallback (T, Y
// untouched).
__global__ void k_surr_apply(int n, double *__restrict__ T, double *__restrict__ Y,
                             const float *__restrict__ pred, long ldp,
                             const float *__restrict__ omean, const float *__restrict__ ostd,
                             const float *__restrict__ oc,
                             const double *__restrict__ proj, const unsigned short *__restrict__ X,
                             float feat_lim, double tol_T, double dT_max,
                             int *__restrict__ flag, double *__restrict__ T_energy) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const int K = CK_NEQ - 1;
  double y0[CK_NEQ - 1], y1[CK_NEQ - 1];
  for (int k = 0; k < K; k++) y0[k] = Y[(long)c * K + k];
  const double T0 = T[c];
  double dT, Te;
  const int bad = surr_decide(y0, T0, pred + (long)c * ldp, omean, ostd, oc, proj,
                              X + (long)c * IZ_SURR_XLD, feat_lim, tol_T, dT_max, y1, dT, Te);
  if (T_energy) T_energy[c] = Te;
  flag[c] = bad;
  if (!bad) {
    T[c] = T0 + dT;
    for (int k = 0; k < K; k++) Y[(long)c * K + k] = y1[k];
  }
}

// pack the flagged cells (order not kept) and return their indices
__global__ void k_surr_gather(int n, const int *__restrict__ flag, const double *__restrict__ T,
                              const double *__restrict__ rho, const double *__restrict__ Y,
                              int *__restrict__ count, int *__restrict__ idx,
                              double *__restrict__ Tw, double *__restrict__ rw,
                              double *__restrict__ Yw) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n || !flag[c]) return;
  const int j = atomicAdd(count, 1);
  idx[j] = c;
  Tw[j] = T[c];
  rw[j] = rho[c];
  for (int k = 0; k < CK_NEQ - 1; k++) Yw[(long)j * (CK_NEQ - 1) + k] = Y[(long)c * (CK_NEQ - 1) + k];
}

__global__ void k_surr_scatter(int m, const int *__restrict__ idx, const double *__restrict__ Tw,
                               const double *__restrict__ Yw, double *__restrict__ T,
                               double *__restrict__ Y) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= m) return;
  const int c = idx[j];
  T[c] = Tw[j];
  for (int k = 0; k < CK_NEQ - 1; k++) Y[(long)c * (CK_NEQ - 1) + k] = Yw[(long)j * (CK_NEQ - 1) + k];
}

__global__ void k_zero_int(int *p) { *p = 0; }

extern "C" int izem_surr_features(izem_ctx *ctx, int n, const double *T, const double *rho,
                                  const double *Y, double dt, const float *mean,
                                  const float *istd, void *X) {
  if (!ctx || !ctx->chem || n < 0 || !T || !rho || !Y || !(dt > 0) || !mean || !istd || !X)
    return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  hipLaunchKernelGGL(k_surr_features, dim3(iz_blocks(n, 256)), dim3(256), 0, ctx->stream, n, T,
                     rho, Y, log(dt), mean, istd, (unsigned short *)X);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_surr_apply(izem_ctx *ctx, int n, double *T, double *Y, const float *pred,
                               long ldp, const float *omean, const float *ostd, const float *oc,
                               const double *proj, const void *X, float feat_lim, double tol_T,
                               double dT_max, int *flag, double *T_energy) {
  if (!ctx || !ctx->chem || n < 0 || !T || !Y || !pred || !omean || !ostd || !oc || !proj ||
      !X || !flag)
    return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  int pk = iz_prof_begin(ctx, IZP_CHEM);
  hipLaunchKernelGGL(k_surr_apply, dim3(iz_blocks(n, 128)), dim3(128), 0, ctx->stream, n, T, Y,
                     pred, ldp, omean, ostd, oc, proj, (const unsigned short *)X, feat_lim, tol_T,
                     dT_max, flag, T_energy);
  iz_prof_end(ctx, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// integrate the flagged cells with the BDF path: gather into the caller's
// work arrays (idx[n], Tw[n], rw[n], Yw[9 n], counter: 1 int), run
// izem_psr_batch on them, scatter back; *nfall receives their number
extern "C" int izem_surr_fallback(izem_ctx *ctx, int n, double *T, const double *rho,
                                  double *Y, double dt, const int *flag, int *counter, int *idx,
                                  double *Tw, double *rw, double *Yw, int *nfall) {
  if (!ctx || !ctx->chem || n < 0 || !T || !rho || !Y || !flag || !counter || !idx || !Tw ||
      !rw || !Yw || !nfall || !(dt > 0))
    return IZEM_E_ARG;
  *nfall = 0;
  if (n == 0) return IZEM_OK;
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, ctx->stream, counter);
  hipLaunchKernelGGL(k_surr_gather, dim3(iz_blocks(n, 256)), dim3(256), 0, ctx->stream, n, flag,
                     T, rho, Y, counter, idx, Tw, rw, Yw);
  int m = 0;
  IZ_CHECK(hipMemcpyAsync(&m, counter, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  IZ_CHECK(hipStreamSynchronize(ctx->stream));
  *nfall = m;
  if (m == 0) return IZEM_OK;
  int r = izem_psr_batch(ctx, m, Tw, rw, Yw, dt, nullptr);
  if (r != IZEM_OK) return r;
  hipLaunchKernelGGL(k_surr_scatter, dim3(iz_blocks(m, 256)), dim3(256), 0, ctx->stream, m, idx,
                     Tw, Yw, T, Y);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// ===================================================================
// The surrogate inside the flow's reaction step: reaction_selec with
// the learned substep on the cells the indicator accepts and the BDF
// reactor kernel on the others.  The dispatch it joins is
// reaction_selec (module_reaction.f90:47-90: DVODE or MIL by
// inp%reac_selec); the surrogate itself has no reference counterpart.
// ===================================================================

// box cell -> flow-array cell (the mapping of k_reaction_queue)
__device__ inline long box_cell(const IzDims &d, const IzBox &b, long cell) {
  const int ni = b.i1 - b.i0 + 1, nj = b.j1 - b.j0 + 1;
  const int i = b.i0 + (int)(cell % ni);
  const long r = cell / ni;
  return iz_cidx(d, i, b.j0 + (int)(r % nj), b.k0 + (int)(r / nj));
}

// feature rows of box cells c0 .. c0 + m - 1 (CHEMKIN units, as the
// reactor kernel converts them)
__global__ void __launch_bounds__(256) k_surr_flow_features(
    IzDims d, IzBox b, long c0, int m, const double *__restrict__ dtp, double scale,
    double time_ref, double T_ref, double rho_cgs, const double *__restrict__ T,
    const double *__restrict__ v, const float *__restrict__ mean, const float *__restrict__ istd,
    unsigned short *__restrict__ X) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= m) return;
  const long c = box_cell(d, b, c0 + j);
  const double rho0 = v[c], rho_i = 1.0 / rho0;
  double y[CK_NEQ - 1];
  for (int l = 0; l < CK_NEQ - 1; l++) y[l] = v[(IZ_NIV + l) * d.nc + c] * rho_i;
  const double dt_phys = (scale * (*dtp)) * time_ref;
  surr_row(T[c] * T_ref, rho0 * rho_cgs, y, log(dt_phys), mean, istd,
           X + (long)j * IZ_SURR_XLD);
}

// the network's substep on box cells c0 .. c0 + m - 1: accepted cells get
// T and rho Y_k as the reactor kernel writes them (clipped Y_k, the last
// species closing the sum) and enter DTmax; rejected cells are appended
// to the fallback list, untouched
__global__ void __launch_bounds__(256) k_surr_flow_apply(
    IzDims d, IzBox b, long c0, int m, const float *__restrict__ pred,
    const float *__restrict__ omean, const float *__restrict__ ostd, const float *__restrict__ oc,
    const double *__restrict__ proj, const unsigned short *__restrict__ X, float feat_lim,
    double tol_T, double dT_max, double T_ref, double *__restrict__ T, double *__restrict__ v,
    int *__restrict__ nfall, int *__restrict__ list, double *__restrict__ ts) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  int reject = 0;
  double dtabs = 0.0;
  if (j < m) {
    const long c = box_cell(d, b, c0 + j);
    const double rho0 = v[c], rho_i = 1.0 / rho0;
    double y0[CK_NEQ - 1], y1[CK_NEQ - 1];
    for (int l = 0; l < CK_NEQ - 1; l++) y0[l] = v[(IZ_NIV + l) * d.nc + c] * rho_i;
    const double T0 = T[c] * T_ref;
    double dT, Te;
    reject = surr_decide(y0, T0, pred + (long)j * 64, omean, ostd, oc, proj,
                         X + (long)j * IZ_SURR_XLD, feat_lim, tol_T, dT_max, y1, dT, Te);
    if (!reject) {
      const double T1 = T0 + dT;
      T[c] = T1 * (1.0 / T_ref);
      dtabs = fabs(T1 - T0);
      double sumY = 0.0;
      for (int l = 0; l < CK_NEQ - 2; l++) {
        const double Ya = fmin(fmax(y1[l], 0.0), 1.0);
        v[(IZ_NIV + l) * d.nc + c] = rho0 * Ya;
        sumY = sumY + Ya;
      }
      v[(IZ_NIV + CK_NEQ - 2) * d.nc + c] = rho0 * (1.0 - sumY);
    }
  }
  // one list reservation per wave
  const unsigned long long mask = __ballot(reject);
  int base = 0;
  if (lane == 0 && mask) base = atomicAdd(nfall, __popcll(mask));
  base = __shfl(base, 0, 64);
  if (reject) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = (int)(c0 + j);
  for (int off = 32; off > 0; off >>= 1) dtabs = fmax(dtabs, __shfl_xor(dtabs, off, 64));
  if (lane == 0) atomic_max_posd(&ts[5], dtabs);
}

__global__ void k_surr_count(unsigned long long *__restrict__ counts, long n,
                             const int *__restrict__ nfall) {
  counts[0] += (unsigned long long)n;
  counts[1] += (unsigned long long)*nfall;
}

extern "C" int izem_surr_attach(izem_ctx *ctx, const izem_surrogate *s, long chunk) {
  if (!ctx || !ctx->chem) return IZEM_E_ARG;
  IzChem *ch = ctx->chem;
  if (!s) {
    IZ_CHECK(hipStreamSynchronize(ctx->stream));
    surr_free(ch->surr);
    ch->surr = nullptr;
    ch->reac_selec = IZEM_REAC_DVODE;
    ch->sel_gen++;
    return IZEM_OK;
  }
  if (chunk < 128 || chunk > (1L << 26)) return IZEM_E_ARG;
  for (int l = 0; l < 4; l++)
    if (!s->Wt[l] || !s->b[l] || (((uintptr_t)s->Wt[l]) & 15)) return IZEM_E_ARG;
  if (!s->in_mean || !s->in_istd || !s->out_mean || !s->out_std || !s->out_c || !s->proj ||
      !(s->feat_lim > 0) || !(s->tol_T >= 0) || s->dT_max != s->dT_max)
    return IZEM_E_ARG;
  const IzBox b = react_box(ctx);
  if (b.n > INT_MAX) return IZEM_E_ARG;
  IZ_CHECK(hipStreamSynchronize(ctx->stream));
  IzSurr *u = ch->surr;
  if (u && (u->chunk != chunk || u->list_cap < b.n)) {
    surr_free(u);
    u = ch->surr = nullptr;
  }
  if (!u) {
    u = (IzSurr *)calloc(1, sizeof(IzSurr));
    if (!u) return IZEM_E_NOMEM;
    u->chunk = chunk;
    u->list_cap = b.n > 0 ? b.n : 1;
    if (hipMalloc(&u->X, chunk * IZ_SURR_XLD * sizeof(unsigned short)) != hipSuccess ||
        hipMalloc(&u->pred, chunk * 64 * sizeof(float)) != hipSuccess ||
        hipMalloc(&u->list, u->list_cap * sizeof(int)) != hipSuccess ||
        hipMalloc(&u->nfall, sizeof(int)) != hipSuccess ||
        hipMalloc(&u->counts, 2 * sizeof(unsigned long long)) != hipSuccess ||
        hipMemset(u->counts, 0, 2 * sizeof(unsigned long long)) != hipSuccess) {
      surr_free(u);
      return IZEM_E_NOMEM;
    }
    ch->surr = u;
  }
  u->d = *s;
  ch->sel_gen++;
  return IZEM_OK;
}

extern "C" int izem_reaction_surrogate(izem_ctx *ctx, const double *dt, double scale, double *T,
                                       double *W_i, double *cp, double *ha, double *v) {
  if (!ctx || !ctx->chem || !dt || !T || !W_i || !cp || !ha || !v) return IZEM_E_ARG;
  IzChem *ch = ctx->chem;
  IzSurr *u = ch->surr;
  if (!u) return IZEM_E_STATE;
  const IzBox b = react_box(ctx);
  const long n = b.n;
  if (n > u->list_cap) return IZEM_E_STATE;
  hipLaunchKernelGGL(k_chem_prep, dim3(1), dim3(1), 0, ctx->stream, ch->counter, ctx->ts, 1);
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, ctx->stream, u->nfall);
  if (n > 0) {
    const double rho_cgs = ctx->o.rho_ref * 1.0e-3;
    const izem_surrogate &sd = u->d;
    for (long c0 = 0; c0 < n; c0 += u->chunk) {
      const int m = (int)((n - c0 < u->chunk) ? n - c0 : u->chunk);
      int pk = iz_prof_begin(ctx, IZP_CHEM);
      hipLaunchKernelGGL(k_surr_flow_features, dim3(iz_blocks(m, 256)), dim3(256), 0,
                         ctx->stream, ctx->d, b, c0, m, dt, scale, ctx->o.time_ref, ctx->o.T_ref,
                         rho_cgs, T, v, sd.in_mean, sd.in_istd, u->X);
      iz_prof_end(ctx, pk);
      int r = izem_mlp_infer(ctx, m, u->X, sd.Wt, sd.b, u->pred);
      if (r) return r;
      pk = iz_prof_begin(ctx, IZP_CHEM);
      hipLaunchKernelGGL(k_surr_flow_apply, dim3(iz_blocks(m, 256)), dim3(256), 0, ctx->stream,
                         ctx->d, b, c0, m, u->pred, sd.out_mean, sd.out_std, sd.out_c, sd.proj,
                         u->X, sd.feat_lim, sd.tol_T, sd.dT_max, ctx->o.T_ref, T, v, u->nfall,
                         u->list, ctx->ts);
      iz_prof_end(ctx, pk);
    }
    // the fallback cells through the reactor kernel (a queue as long as
    // the list, read on the device)
    int pk = iz_prof_begin(ctx, IZP_CHEM);
    // the list's length is on the device: full waves over the whole chip
    int lanes;
    const int grid = persistent_grid(ctx, n, &lanes);
    reaction_queue(ctx, b, dim3(grid), 64, dt, scale, T, v, u->list, u->nfall);
    iz_prof_end(ctx, pk);
    ch->order_n = 0;
    hipLaunchKernelGGL(k_surr_count, dim3(1), dim3(1), 0, ctx->stream, u->counts, n, u->nfall);
    IZ_CHECK(hipGetLastError());
  }
  return reaction_tail(ctx, dt, scale, T, W_i, cp, ha, v);
}

extern "C" int izem_reac_selec(izem_ctx *ctx, int solver) {
  if (!ctx || !ctx->chem || solver < IZEM_REAC_DVODE || solver > IZEM_REAC_SURROGATE)
    return IZEM_E_ARG;
  if (solver == IZEM_REAC_SURROGATE && !ctx->chem->surr) return IZEM_E_STATE;
  ctx->chem->reac_selec = solver;
  ctx->chem->sel_gen++;
  return IZEM_OK;
}

extern "C" int izem_reaction_selec(izem_ctx *ctx, const double *dt, double scale, double *T,
                                   double *W_i, double *cp, double *ha, double *v) {
  if (!ctx || !ctx->chem) return IZEM_E_ARG;
  if (ctx->chem->reac_selec == IZEM_REAC_SURROGATE)
    return izem_reaction_surrogate(ctx, dt, scale, T, W_i, cp, ha, v);
  return izem_reaction_dvode(ctx, dt, scale, T, W_i, cp, ha, v);
}

extern "C" int izem_surr_counts(izem_ctx *ctx, unsigned long long out[2]) {
  if (!ctx || !ctx->chem || !out) return IZEM_E_ARG;
  IzSurr *u = ctx->chem->surr;
  if (!u) return IZEM_E_STATE;
  IZ_CHECK(hipMemcpyAsync(out, u->counts, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                          ctx->stream));
  IZ_CHECK(hipStreamSynchronize(ctx->stream));
  IZ_CHECK(hipMemset(u->counts, 0, 2 * sizeof(unsigned long long)));
  return IZEM_OK;
}
