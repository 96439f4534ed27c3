// sedcol_kernels.hip -- gfx950 kernels of the sediment-column hot path.
//
// One column per lane group (LPC lanes, lane = layer, all 11 state
// variables in VGPRs); a 256-thread block holds 256/LPC columns.  Wet columns
// are binned by K into LPC = 16/32/64 lists so a group never wastes more than
// half its lanes.  Fixed-step methods keep the state in registers for a
// whole window of steps; the adaptive EMP kernel keeps it for the whole
// integration span and every forcing record inside it.
//
// Top fluxes are produced on lane 0 (one value per variable and stage); they
// are staged in LDS and accumulated by lanes 0..NV-1, lane n owning
// variable n, so no lane carries per-variable flux registers.
#include <atomic>

#include "sedcol_kernels.hpp"

namespace sc {

constexpr int BLOCK = 256;

// ---------------------------------------------------------------------------
// per-lane set-up
// ---------------------------------------------------------------------------

struct Geo {
  double phiI, bfac, B;
};

__device__ __forceinline__ void setup_lane(const Dev &d, int c, int l, Lane &L, Geo &G, long long &cell)
{
  const int o = d.off[c];
  L.l = l;
  L.K = d.off[c + 1] - o;
  L.active = l < L.K;
  cell = (long long)o + l;
  L.dz = L.active ? d.dz[cell] : 1.0;
  L.dzc = L.active ? (l > 0 ? d.dzc[cell] : L.dz) : 1.0;
  L.phi = L.active ? d.phi[cell] : 0.5;
  G.phiI = L.active ? d.phiI[cell] : 0.5;
  L.cap = (L.active && d.fcap) ? d.fcap[cell] : 0.0;
  L.ze1 = (L.active && d.zw.on) ? d.zw.e1[cell] : 1.0;
  L.ze2 = (L.active && d.zw.on) ? d.zw.e2[cell] : 1.0;
  L.zcum = d.zw.on ? d.zw.cum[c] : 1.0;
  G.bfac = L.active ? d.bfac[cell] : 0.0;
  G.B = d.biot[c];
}

// whether b holds on any active lane of the group: the group's bits of the
// wave's ballot, instead of a reduction over the lanes
template <int LPC>
__device__ __forceinline__ bool group_any(bool b)
{
  const unsigned long long m = __ballot(b);
  if constexpr (LPC == 64) {
    return m != 0;
  } else {
    const unsigned lane = __lane_id();
    const unsigned half = (lane & 32u) ? (unsigned)(m >> 32) : (unsigned)m;
    if constexpr (LPC == 32) return half != 0;
    else return ((lane & 16u) ? half >> 16 : half & 0xffffu) != 0;
  }
}

// load forcing record r of column c: bottom-water concentrations and top
// fluxes (0 for a closed top) to the group's LDS slot, temperature-dependent
// coefficients to L
__device__ __forceinline__ bool load_top(const Dev &d, const sedcol_params &p, int c, int r, int n, double *sbc)
{
  const int bc = part(n) ? p.bcup_part : p.bcup_dis;
  const double w = d.cbw[((long long)r * NV + n) * d.ncol + c];
  const double f = d.fup[(long long)r * d.fup_rec_stride + (long long)n * d.ncol + c];
  const double t = (bc == 1 || bc == 4) ? f : 0.0;
  sbc[n] = w;
  sbc[NV + n] = t;
  return in_range(w, kStateLo, kStateHi) && in_range(t, kStateLo, kStateHi);
}

template <int LPC, int ARITH>
__device__ __forceinline__ void load_forcing(const Dev &d, const sedcol_params &p, int c, int r, const Geo &G,
                                             Lane &L, double *sbc)
{
  bool ok = true;
  if (L.l < NV) ok = load_top(d, p, c, r, L.l, sbc);
  const double T = d.temp[(long long)r * d.ncol + c];
  diffusivities<ARITH>(p, G.B, T, G.phiI, G.bfac, L);
  if (ARITH == ARITH_REF) {
    ok = ok && params_ok(p) && (!L.active || lane_ok(L));
    L.wide = group_any<LPC>(!ok);
  }
}

// The boundary values of a group's slot in registers: of each variable the one
// that its boundary condition uses (column_terms with TF = 0).
__device__ __forceinline__ void take_top(const sedcol_params &p, const double *sbc, double (&bc)[NV])
{
#pragma unroll
  for (int n = 0; n < NV; ++n) bc[n] = sbc[(part(n) ? p.bcup_part : p.bcup_dis) != 2 ? NV + n : n];
}

// top fluxes of one right-hand side, held by the group's first lane, into the
// group's LDS slot: one branch for all variables
__device__ __forceinline__ void store_top(bool first, const double (&Ft)[NV], double *F)
{
  if (first) {
#pragma unroll
    for (int n = 0; n < NV; ++n) F[n] = Ft[n];
  }
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// single right-hand side (get_rhs) for parity and diagnostics
// ---------------------------------------------------------------------------

template <int LPC, int ARITH>
__global__ __launch_bounds__(BLOCK) void k_rhs(Dev d, const int *list, int nlist, sedcol_params p, int rec,
                                               const double *conc, double *rhs, double *flux, double *sinks)
{
  constexpr int G = BLOCK / LPC;
  __shared__ double sbc[G][2 * NV];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  const bool valid = slot < nlist;
  const int c = valid ? list[slot] : 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  if (valid) {
    setup_lane(d, c, l, L, Gm, cell);
    load_forcing<LPC, ARITH>(d, p, c, rec, Gm, L, sbc[g]);
  }
  __syncthreads();
  if (!valid) return;
  double x[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) x[n] = L.active ? conc[n * d.ncell + cell] : 0.0;
  double sC, sN;
  column_rhs<LPC, ARITH>(p, L, sbc[g], x, sC, sN, [&](int n, double r, double F) {
    if (L.active && rhs) rhs[n * d.ncell + cell] = r;
    if (l == 0 && flux) flux[(long long)n * d.ncol + c] = F;
  }, &d.zw);
  if (L.active && sinks) {
    sinks[cell] = sC;
    sinks[d.ncell + cell] = sN;
  }
}

// ---------------------------------------------------------------------------
// fixed-step window: EULER, RK4, RK4 3/8, EMP-1, EMP-2
// ---------------------------------------------------------------------------

// Instances that take a little more than the 256 registers of two waves per
// SIMD.  A launch of at most one wave per SIMD is a lone chain per wave, which
// the registers suit best; beyond, the second wave hides more than the few
// spilled values cost (FULL).  24 steps of 30 layers, one wave and two:
//                                   600 columns     2200 columns    20000 columns
//   EMP-2, reference form           210    216 us   381    296 us   1808   1283 us
//   EMP-1 ext. form                 168    172      296    227      1345    937
//   EMP-1 geometric, fast form      158    168      279    223      1262    921
// The Euler step of the extended form gains from two waves at every size (600
// columns 138 -> 131 us, 20000 columns 1025 -> 699 us).
constexpr bool fixed_split(int method, int arith, int pw)
{
  return method == SEDCOL_EMP2   ? arith == ARITH_REF && pw == 0
         : method == SEDCOL_EMP1 ? (arith == ARITH_EXT && pw == 0) || (arith == ARITH_FAST && pw == 1)
                                 : false;
}
constexpr int fixed_waves(int method, int arith, bool full)
{
  return full || (method == SEDCOL_EULER && arith == ARITH_EXT) ? 2 : 1;
}

template <int LPC, int METHOD, int ARITH, int PW, bool FULL>
__global__ __launch_bounds__(BLOCK, fixed_waves(METHOD, ARITH, FULL)) void k_fixed(Dev d, const int *list, int nlist,
                                                                                 sedcol_params p, int rec, double dt,
                                                                                 int nsteps, int *errflag)
{
  constexpr int G = BLOCK / LPC;
  __shared__ double sbc[G][2 * NV];
  __shared__ double sF[G][4][NV];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  const bool valid = slot < nlist;
  const int c = valid ? list[slot] : 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  if (valid) {
    setup_lane(d, c, l, L, Gm, cell);
    load_forcing<LPC, ARITH>(d, p, c, rec, Gm, L, sbc[g]);
  }
  __syncthreads();
  if (!valid) return;
  // the boundary values stay in registers for the whole run: read from LDS in
  // every right-hand side, they cost a lone wave 1600 of 4900 cycles.  The two
  // waves of a full EMP-1 launch read them (in registers, 80 and 156 instead of
  // 20 and 80 bytes of scratch, and 4 and 16 % more time at 20000 columns)
  constexpr int TF = FULL && METHOD == SEDCOL_EMP1 ? NV : 0;
  double bcr[NV];
  const double *bc = sbc[g];
  if constexpr (TF == 0) {
    take_top(p, sbc[g], bcr);
    bc = bcr;
  }
  double(*F)[NV] = sF[g];
  const bool act = L.active;
  const bool own = l < NV;  // lane l accumulates the top flux of variable l

  double x[NV];
  const double *from = d.hconc ? d.hconc : d.conc;
#pragma unroll
  for (int n = 0; n < NV; ++n) x[n] = act ? from[n * d.ncell + cell] : 0.0;
  double fint = own ? d.colacc[(long long)l * d.ncol + c] : 0.0;
  double fintc = own ? d.colacc[(long long)(NV + l) * d.ncol + c] : 0.0;
  double flast = own ? d.flux[(long long)l * d.ncol + c] : 0.0;
  double acc[5], accc[5];
#pragma unroll
  for (int a = 0; a < 5; ++a) {
    acc[a] = act ? d.cellacc[a * d.ncell + cell] : 0.0;
    accc[a] = act ? d.cellacc[(5 + a) * d.ncell + cell] : 0.0;
  }
  sedcol_coldiag dg = d.diag[c];
  int64_t zs = 0;
  const double third = 1.0 / 3.0;

  for (int s = 0; s < nsteps; ++s) {
    double sC, sN, Ft[NV];
    if (METHOD == SEDCOL_EULER) {
      double r0[NV];
      column_rhs<LPC, ARITH, TF>(p, L, bc, x, sC, sN, [&](int n, double r, double Fv) {
        r0[n] = r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[0]);
#pragma unroll
      for (int n = 0; n < NV; ++n) x[n] = x[n] + dt * r0[n];
      if (own) {
        kadd(fint, fintc, dt * F[0][l]);
        flast = F[0][l];
      }
      kadd(acc[0], accc[0], dt * sC);
      kadd(acc[1], accc[1], dt * sN);
    } else if (METHOD == SEDCOL_RUNGE_KUTTA_4) {
      // solver_library.F90:142-163
      double cs[NV], k[NV];
      double aC, aN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, x, sC, sN, [&](int n, double r, double Fv) {
        k[n] = 0.5 * r;
        cs[n] = x[n] + (0.5 * dt) * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[0]);
      aC = 0.5 * sC;
      aN = 0.5 * sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        k[n] = k[n] + r;
        cs[n] = x[n] + (0.5 * dt) * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[1]);
      aC = aC + sC;
      aN = aN + sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        k[n] = k[n] + r;
        cs[n] = x[n] + dt * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[2]);
      aC = aC + sC;
      aN = aN + sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        k[n] = k[n] + 0.5 * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[3]);
      aC = aC + 0.5 * sC;
      aN = aN + 0.5 * sN;
      const double w = dt * third;
#pragma unroll
      for (int n = 0; n < NV; ++n) x[n] = x[n] + w * k[n];
      if (own) {
        kadd(fint, fintc, w * (((0.5 * F[0][l] + F[1][l]) + F[2][l]) + 0.5 * F[3][l]));
        flast = F[3][l];
      }
      kadd(acc[0], accc[0], w * aC);
      kadd(acc[1], accc[1], w * aN);
    } else if (METHOD == SEDCOL_RUNGE_KUTTA_4_38) {
      // solver_library.F90:164-185
      double cs[NV], k1[NV], k2[NV];
      double s1C, s1N, s2C, s2N;
      column_rhs<LPC, ARITH, TF>(p, L, bc, x, sC, sN, [&](int n, double r, double Fv) {
        k1[n] = r;
        cs[n] = x[n] + (third * dt) * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[0]);
      s1C = sC;
      s1N = sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        k2[n] = r;
        cs[n] = x[n] + dt * (r - third * k1[n]);
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[1]);
      s2C = sC;
      s2N = sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        cs[n] = x[n] + dt * ((k1[n] - k2[n]) + r);
        k1[n] = (k1[n] + 3.0 * k2[n]) + 3.0 * r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[2]);
      double aC = (s1C + 3.0 * s2C) + 3.0 * sC;
      double aN = (s1N + 3.0 * s2N) + 3.0 * sN;
      column_rhs<LPC, ARITH, TF>(p, L, bc, cs, sC, sN, [&](int n, double r, double Fv) {
        k1[n] = k1[n] + r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[3]);
      aC = aC + sC;
      aN = aN + sN;
      const double w = (dt * 1.0) / 8.0;
#pragma unroll
      for (int n = 0; n < NV; ++n) x[n] = x[n] + w * k1[n];
      if (own) {
        kadd(fint, fintc, w * (((F[0][l] + 3.0 * F[1][l]) + 3.0 * F[2][l]) + F[3][l]));
        flast = F[3][l];
      }
      kadd(acc[0], accc[0], w * aC);
      kadd(acc[1], accc[1], w * aN);
    } else {  // EMP-1 / EMP-2 with a fixed step
      double f0[NV];
      column_rhs<LPC, ARITH, TF>(p, L, bc, x, sC, sN, [&](int n, double r, double Fv) {
        f0[n] = r;
        Ft[n] = Fv;
      }, &d.zw);
      store_top(l == 0, Ft, F[0]);
      const double p1 = pfactor<LPC, false, PW>(x, f0, x, dt, act, zs, dg.newton);
      if (p1 < dg.p_min) dg.p_min = p1;
      if (METHOD == SEDCOL_EMP1) {
#pragma unroll
        for (int n = 0; n < NV; ++n) x[n] = x[n] + (dt * p1) * f0[n];
        if (own) {
          kadd(fint, fintc, (dt * p1) * F[0][l]);
          flast = F[0][l];
        }
        kadd(acc[0], accc[0], (dt * p1) * sC);
        kadd(acc[1], accc[1], (dt * p1) * sN);
      } else {
        double c1[NV];
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const double y = x[n] + (dt * p1) * f0[n];
          c1[n] = y < 0.0 ? 0.0 : y;
        }
        const double s0C = sC, s0N = sN;
        column_rhs<LPC, ARITH, TF>(p, L, bc, c1, sC, sN, [&](int n, double r, double Fv) {
          f0[n] = (f0[n] + r) * 0.5;
          Ft[n] = Fv;
        }, &d.zw);
      store_top(l == 0, Ft, F[1]);
        const double p2 = pfactor<LPC, true, PW>(x, f0, c1, dt, act, zs, dg.newton);
        if (p2 < dg.p_min) dg.p_min = p2;
#pragma unroll
        for (int n = 0; n < NV; ++n) x[n] = x[n] + (dt * p2) * f0[n];
        if (own) {
          kadd(fint, fintc, (dt * p2) * ((F[0][l] + F[1][l]) * 0.5));
          flast = F[1][l];
        }
        kadd(acc[0], accc[0], (dt * p2) * ((s0C + sC) * 0.5));
        kadd(acc[1], accc[1], (dt * p2) * ((s0N + sN) * 0.5));
      }
    }
    dg.accepted += 1;
    dg.dt_last = dt;
    if (dt < dg.dt_minacc) dg.dt_minacc = dt;
    // clamp: Patankar rounding guard (EMP), or the callers' minimum clamp;
    // one test for negative values and NaN, most steps have neither
    bool odd = false;
#pragma unroll
    for (int n = 0; n < NV; ++n) odd |= !(x[n] >= 0.0);
    if (__any(odd)) {
      if (METHOD >= SEDCOL_EMP1 || p.clamp) {
#pragma unroll
        for (int n = 0; n < NV; ++n)
          if (x[n] < 0.0) {
            if (elem(n) >= 0) kadd(acc[2 + elem(n)], accc[2 + elem(n)], 0.0 - x[n]);
            x[n] = 0.0;
          }
      }
      bool nan = false;
#pragma unroll
      for (int n = 0; n < NV; ++n) nan |= act && (x[n] != x[n]);
      if (group_any<LPC>(nan)) {
        dg.status = 1;
        if (l == 0) {
          atomicOr(errflag, 1);
          if (d.hflag) *d.hflag = 1;
        }
        break;
      }
    }
  }

#pragma unroll
  for (int n = 0; n < NV; ++n)
    if (act) d.conc[n * d.ncell + cell] = x[n];
  if (own) {
    d.colacc[(long long)l * d.ncol + c] = fint;
    d.colacc[(long long)(NV + l) * d.ncol + c] = fintc;
    d.flux[(long long)l * d.ncol + c] = flast;
  }
  if (d.hconc) {
#pragma unroll
    for (int n = 0; n < NV; ++n)
      if (act) d.hconc[n * d.ncell + cell] = x[n];
    if (own) d.hflux[(long long)l * d.ncol + c] = flast;
  }
#pragma unroll
  for (int a = 0; a < 5; ++a)
    if (act) {
      d.cellacc[a * d.ncell + cell] = acc[a];
      d.cellacc[(5 + a) * d.ncell + cell] = accc[a];
    }
  const double zsum = lg_sum<LPC>((double)zs);
  if (l == 0) {
    dg.zero_sink += (int64_t)zsum;
    d.diag[c] = dg;
  }
}

// ---------------------------------------------------------------------------
// adaptive EMP: per-column step size, persistent over [t_start, t_end)
// ---------------------------------------------------------------------------

// minimum waves per SIMD requested from the register allocator: 2 fits the
// adaptive step in 256 VGPRs without scratch (1 lets it take 256 + AGPRs,
// 3 spills about 340 bytes per lane).  With geometric weights the step does not
// fit (130 to 190 bytes of scratch per lane) and one wave is faster, reference
// form, 1 h: 1201 columns of 30 to 60 layers 157 -> 104 ms, 9000 columns of 10 to
// 60 layers 300 -> 235 ms.  It then has room for the boundary values and the
// solve's coefficients, which were read from LDS in every evaluation (3 h of the
// 1201 columns 273 -> 264 ms).  Many columns of long bins only, reference form,
// 15 min, were faster in two waves before the right-hand side became one stretch
// of code: 12000 of 34 to 60 layers 128, now 133 ms, 25000 of them 257, now 276.
// Two waves of the present code spill 172 to 232 bytes: 144 and 288 ms, without
// the quotients by reciprocals 135 and 265.
#ifndef SEDCOL_EMP_MIN_WAVES
#define SEDCOL_EMP_MIN_WAVES 2
#endif
#ifndef SEDCOL_GEO_MIN_WAVES
#define SEDCOL_GEO_MIN_WAVES 1
#endif

// Work-queue kernel: a grid sized to the resident capacity, each lane group
// taking the next column from *next (atomic counter) when it finishes one,
// so columns needing many steps do not leave other lanes idle.  Every column
// is integrated over [t_start, t_end) record by record (record r covers
// [t0 + r dt_rec, t0 + (r+1) dt_rec), the first and last extend outward),
// with its own step size carried in diag.dt_next.  Each group exits when the
// queue is empty, so every wave reaches the end.
//
// Windows: with ctl.window > 0 a column stops after that many attempts in
// one launch and saves its position (record, time left in the record,
// attempts so far) in d.wrec / d.wrem / d.watt; *pending counts the columns
// so stopped.  With ctl.resume = 1 every column continues from its saved
// position (k_emp_begin sets the start position) and columns whose record
// is past r1 are skipped.  A column's operations are the same however its
// attempts are split over launches, so windowed and single-launch runs give
// identical results.
template <int LPC, int ARITH, int BLK, int PW>
__global__ __launch_bounds__(BLK, PW == 1 ? SEDCOL_GEO_MIN_WAVES : SEDCOL_EMP_MIN_WAVES) void k_emp_adaptive(
    const Dev *dptr, const int *list, int nlist, const sedcol_params *__restrict__ pptr,
    const EmpCtl *__restrict__ cptr, int *next, int *pending, int *work, int *errflag)
{
  // Domain, parameters and span are read through pointers to device copies
  // rather than passed by value: about 100 dwords of by-value arguments would
  // be held in SGPRs for the whole kernel and spill.
  const Dev &d = *dptr;
  const sedcol_params &p = *pptr;
  const EmpCtl &ctl = *cptr;
  constexpr int G = BLK / LPC;
  __shared__ double sbc[G][2 * NV];
  __shared__ double sF[G][2][NV];
  __shared__ int sslot[G];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const bool own = l < NV;  // lane l accumulates the top flux of variable l
  double(*F)[NV] = sF[g];
  // one wave per SIMD (PW == 1) has room for the boundary values in registers
  constexpr int TF = PW == 1 ? 0 : NV;
  double bcr[NV];
  const double *bc = sbc[g];
  if constexpr (PW == 1) bc = bcr;
  auto boundary = [&]() {
    __builtin_amdgcn_wave_barrier();
    if constexpr (PW == 1) take_top(p, sbc[g], bcr);
  };
  const int r1 = ctl.r1;

  // state of the group's current column
  int c = 0, r = 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  double x[NV];
  // Per-lane budget sums (with their compensations) and the last top flux:
  // touched only when an attempt is accepted, so they live in LDS and leave
  // the registers to the right-hand side.
  __shared__ double sacc[7][BLK];
  double &sinkC = sacc[0][threadIdx.x], &sinkN = sacc[1][threadIdx.x], &fint = sacc[2][threadIdx.x];
  double &sinkCc = sacc[3][threadIdx.x], &sinkNc = sacc[4][threadIdx.x], &fintc = sacc[5][threadIdx.x];
  double &flast = sacc[6][threadIdx.x];
  sedcol_coldiag dg;
  int64_t zs = 0;
  long long attempts = 0;
  int wn = 0;
  double dt = 0.0, rem = 0.0;
  bool have = false, act = false;

  for (;;) {
    if (!have) {
      if (l == 0) sslot[g] = atomicAdd(next, 1);
      __builtin_amdgcn_wave_barrier();
      const int s = sslot[g];
      __builtin_amdgcn_wave_barrier();
      if (s >= nlist) break;
      c = list[s];
      if (ctl.resume) {
        r = d.wrec[c];
        if (r > r1) continue;  // finished in an earlier window
        rem = d.wrem[c];
        attempts = d.watt[c];
      } else {
        r = ctl.r0 - 1;
        rem = 0.0;
        attempts = 0;
      }
      setup_lane(d, c, l, L, Gm, cell);
      act = L.active;
#pragma unroll
      for (int n = 0; n < NV; ++n) x[n] = act ? d.conc[n * d.ncell + cell] : 0.0;
      sinkC = act ? d.cellacc[cell] : 0.0;
      sinkN = act ? d.cellacc[d.ncell + cell] : 0.0;
      sinkCc = act ? d.cellacc[5 * d.ncell + cell] : 0.0;
      sinkNc = act ? d.cellacc[6 * d.ncell + cell] : 0.0;
      fint = own ? d.colacc[(long long)l * d.ncol + c] : 0.0;
      fintc = own ? d.colacc[(long long)(NV + l) * d.ncol + c] : 0.0;
      flast = own ? d.flux[(long long)l * d.ncol + c] : 0.0;
      dg = d.diag[c];
      dt = dg.dt_next;
      if (!(dt > 0.0)) dt = p.emp_dt_max;
      zs = 0;
      wn = 0;
      have = true;
      if (rem > 0.0) {
        // resumed inside record r
        load_forcing<LPC, ARITH>(d, p, c, r, Gm, L, sbc[g]);
        boundary();
      }
    }
    bool finish = false;
    if (!(rem > 0.0)) {
      // next forcing record with a positive span, or the column is done
      ++r;
      if (r > r1) {
        finish = true;
      } else {
        const double lo = (r == 0) ? -INFINITY : d.t0 + (double)r * d.dt_rec;
        const double hi = (r == d.nrec - 1) ? INFINITY : d.t0 + (double)(r + 1) * d.dt_rec;
        const double a = ctl.t_start > lo ? ctl.t_start : lo;
        const double b = ctl.t_end < hi ? ctl.t_end : hi;
        rem = b - a;
        load_forcing<LPC, ARITH>(d, p, c, r, Gm, L, sbc[g]);
        boundary();
        continue;
      }
    }
    bool pause = false;
    if (!finish) {
      if (attempts >= ctl.max_attempts) {
        dg.status = 2;
        if (l == 0) atomicOr(errflag, 2);
        finish = true;
      } else if (ctl.window > 0 && wn >= ctl.window) {
        pause = true;
      }
    }
    if (!finish && !pause) {
      ++attempts;
      ++wn;
      const bool clipped = !(dt < rem);
      const double h = clipped ? rem : dt;
      double f0[NV], c1[NV];
      double s0C, s0N, s1C, s1N;
      column_rhs<LPC, ARITH, TF>(p, L, bc, x, s0C, s0N, [&](int n, double rr, double Fv) {
        f0[n] = rr;
        if (l == 0) F[0][n] = Fv;
      }, &d.zw);
      const double p1 = pfactor<LPC, false, PW>(x, f0, x, h, act, zs, dg.newton);
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const double y = x[n] + (h * p1) * f0[n];
        c1[n] = y < 0.0 ? 0.0 : y;
      }
      column_rhs<LPC, ARITH, TF>(p, L, bc, c1, s1C, s1N, [&](int n, double rr, double Fv) {
        f0[n] = (f0[n] + rr) * 0.5;
        if (l == 0) F[1][n] = Fv;
      }, &d.zw);
      const double p2 = pfactor<LPC, true, PW>(x, f0, c1, h, act, zs, dg.newton);
      // err = max |c2 - c1| / sc: the lane's largest ratio by
      // cross-multiplication over the variables, one division, then the
      // maximum over the layers
      double bn = 0.0, bd = 1.0;
      bool bad = false;
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const double y = x[n] + (h * p2) * f0[n];
        const double yp = vmax(y, 0.0);
        const double sc = p.emp_atol + p.emp_rtol * vmax(yp, x[n]);
        const double dv = fabs(yp - c1[n]);
        // a NaN in y (vmax drops it) or in dv (two infinities), in one comparison
        bad |= __builtin_isunordered(y, dv) || (sc != sc);
        if (dv * bd > bn * sc) {
          bn = dv;
          bd = sc;
        }
      }
      double el = bn / bd;
      bad |= el != el;
      if (!act) {
        el = 0.0;
        bad = false;
      }
      const double err = lg_max<LPC>(el);
      if (group_any<LPC>(bad)) {
        dg.status = 1;
        if (l == 0) atomicOr(errflag, 1);
        finish = true;
      } else {
        const bool accept = (err <= 1.0) || !(h > p.emp_dt_min);
        double fac = err > 0.0 ? 0.9 * drsqrt(err) : 5.0;
        if (fac < 0.2) fac = 0.2;
        if (fac > 5.0) fac = 5.0;
        if (p1 < dg.p_min) dg.p_min = p1;
        if (p2 < dg.p_min) dg.p_min = p2;
        if (accept) {
#pragma unroll
          for (int n = 0; n < NV; ++n) {
            double y = x[n] + (h * p2) * f0[n];
            if (y < 0.0) {
              // rounding guard; rare, so accumulated straight into the
              // lane's own cell of the budget array
              if (elem(n) >= 0 && act)
                kadd(d.cellacc[(2 + elem(n)) * d.ncell + cell], d.cellacc[(7 + elem(n)) * d.ncell + cell], 0.0 - y);
              y = 0.0;
            }
            x[n] = y;
          }
          if (own) {
            kadd(fint, fintc, (h * p2) * ((F[0][l] + F[1][l]) * 0.5));
            flast = F[1][l];
          }
          kadd(sinkC, sinkCc, (h * p2) * ((s0C + s1C) * 0.5));
          kadd(sinkN, sinkNc, (h * p2) * ((s0N + s1N) * 0.5));
          rem = rem - h;
          dg.accepted += 1;
          if (err > 1.0) dg.forced += 1;
          dg.dt_last = h;
          if (h < dg.dt_minacc) dg.dt_minacc = h;
          const double prop = h * fac;
          dt = (clipped && dt > prop) ? dt : prop;
        } else {
          dg.rejected += 1;
          dt = h * fac;
        }
        if (dt < p.emp_dt_min) dt = p.emp_dt_min;
        if (dt > p.emp_dt_max) dt = p.emp_dt_max;
      }
    }
    if (finish || pause) {
#pragma unroll
      for (int n = 0; n < NV; ++n)
        if (act) d.conc[n * d.ncell + cell] = x[n];
      if (act) {
        d.cellacc[cell] = sinkC;
        d.cellacc[d.ncell + cell] = sinkN;
        d.cellacc[5 * d.ncell + cell] = sinkCc;
        d.cellacc[6 * d.ncell + cell] = sinkNc;
      }
      if (own) {
        d.colacc[(long long)l * d.ncol + c] = fint;
        d.colacc[(long long)(NV + l) * d.ncol + c] = fintc;
        d.flux[(long long)l * d.ncol + c] = flast;
      }
      const double zsum = lg_sum<LPC>((double)zs);
      if (l == 0) {
        dg.zero_sink += (int64_t)zsum;
        dg.dt_next = dt;
        d.diag[c] = dg;
        work[c] = attempts < 0x7fffffffll ? (int)attempts : 0x7fffffff;
        // finished (or stopped by an error): record past r1
        d.wrec[c] = pause ? r : r1 + 1;
        d.wrem[c] = rem;
        d.watt[c] = attempts;
        if (pause) atomicAdd(pending, 1);
      }
      have = false;
    }
  }
}

// ---------------------------------------------------------------------------
// adaptive EMP with two layers per lane
// ---------------------------------------------------------------------------
//
// k_emp_adaptive with lane l of a group holding layers 2l and 2l+1
// (column_rhs2, psolve2): a group of LPC lanes takes columns of up to 2 LPC
// layers, so a wave holds twice the columns at the same lane count per
// layer.  Product weights, reference and fast forms.  Every operation per
// layer and every reduction tree are those of k_emp_adaptive, so the
// results are bitwise the same.  LPC >= 16: lanes 0..NV-1 own the top-flux
// accumulators.

// one wave per SIMD: two layers of state and stage values per lane exceed
// the 256 registers of two waves
#ifndef SEDCOL_EMP2_MIN_WAVES
#define SEDCOL_EMP2_MIN_WAVES 1
#endif

__device__ __forceinline__ void setup_lane2(const Dev &d, int c, int l, Lane (&L)[2], Geo (&G)[2],
                                            long long (&cell)[2])
{
  setup_lane(d, c, 2 * l, L[0], G[0], cell[0]);
  setup_lane(d, c, 2 * l + 1, L[1], G[1], cell[1]);
}

template <int ARITH>
__device__ __forceinline__ void load_forcing2(const Dev &d, const sedcol_params &p, int c, int r, int l,
                                              const Geo (&G)[2], Lane (&L)[2], double *sbc)
{
  if (l < NV) (void)load_top(d, p, c, r, l, sbc);
  const double T = d.temp[(long long)r * d.ncol + c];
  diffusivities<ARITH>(p, G[0].B, T, G[0].phiI, G[0].bfac, L[0]);
  diffusivities<ARITH>(p, G[1].B, T, G[1].phiI, G[1].bfac, L[1]);
}

template <int LPC, int ARITH, int BLK>
__global__ __launch_bounds__(BLK, SEDCOL_EMP2_MIN_WAVES) void k_emp_adaptive2(
    const Dev *dptr, const int *list, int nlist, const sedcol_params *__restrict__ pptr,
    const EmpCtl *__restrict__ cptr, int *next, int *pending, int *work, int *errflag)
{
  static_assert(LPC >= 16, "lanes 0..NV-1 own the top-flux accumulators");
  const Dev &d = *dptr;
  const sedcol_params &p = *pptr;
  const EmpCtl &ctl = *cptr;
  constexpr int G = BLK / LPC;
  __shared__ double sbc[G][2 * NV];
  __shared__ double sF[G][2][NV];
  __shared__ int sslot[G];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const bool own = l < NV;
  double(*F)[NV] = sF[g];
  const double *bc = sbc[g];
  const int r1 = ctl.r1;

  int c = 0, r = 0;
  Lane L[2];
  Geo Gm[2];
  long long cell[2] = {0, 0};
  bool act[2] = {false, false};
  double x[2][NV];
  // per-cell budget sums and compensations of both sub-layers, and the
  // lane's top-flux accumulators, in LDS as in k_emp_adaptive
  __shared__ double scell[4][2][BLK];
  __shared__ double scol[3][BLK];
  double &fint = scol[0][threadIdx.x], &fintc = scol[1][threadIdx.x], &flast = scol[2][threadIdx.x];
  sedcol_coldiag dg;
  int64_t zs = 0;
  long long attempts = 0;
  int wn = 0;
  double dt = 0.0, rem = 0.0;
  bool have = false;

  for (;;) {
    if (!have) {
      if (l == 0) sslot[g] = atomicAdd(next, 1);
      __builtin_amdgcn_wave_barrier();
      const int sl = sslot[g];
      __builtin_amdgcn_wave_barrier();
      if (sl >= nlist) break;
      c = list[sl];
      if (ctl.resume) {
        r = d.wrec[c];
        if (r > r1) continue;
        rem = d.wrem[c];
        attempts = d.watt[c];
      } else {
        r = ctl.r0 - 1;
        rem = 0.0;
        attempts = 0;
      }
      setup_lane2(d, c, l, L, Gm, cell);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        act[s] = L[s].active;
#pragma unroll
        for (int n = 0; n < NV; ++n) x[s][n] = act[s] ? d.conc[n * d.ncell + cell[s]] : 0.0;
        scell[0][s][threadIdx.x] = act[s] ? d.cellacc[cell[s]] : 0.0;
        scell[1][s][threadIdx.x] = act[s] ? d.cellacc[d.ncell + cell[s]] : 0.0;
        scell[2][s][threadIdx.x] = act[s] ? d.cellacc[5 * d.ncell + cell[s]] : 0.0;
        scell[3][s][threadIdx.x] = act[s] ? d.cellacc[6 * d.ncell + cell[s]] : 0.0;
      }
      fint = own ? d.colacc[(long long)l * d.ncol + c] : 0.0;
      fintc = own ? d.colacc[(long long)(NV + l) * d.ncol + c] : 0.0;
      flast = own ? d.flux[(long long)l * d.ncol + c] : 0.0;
      dg = d.diag[c];
      dt = dg.dt_next;
      if (!(dt > 0.0)) dt = p.emp_dt_max;
      zs = 0;
      wn = 0;
      have = true;
      if (rem > 0.0) {
        load_forcing2<ARITH>(d, p, c, r, l, Gm, L, sbc[g]);
        __builtin_amdgcn_wave_barrier();
      }
    }
    bool finish = false;
    if (!(rem > 0.0)) {
      ++r;
      if (r > r1) {
        finish = true;
      } else {
        const double lo = (r == 0) ? -INFINITY : d.t0 + (double)r * d.dt_rec;
        const double hi = (r == d.nrec - 1) ? INFINITY : d.t0 + (double)(r + 1) * d.dt_rec;
        const double a = ctl.t_start > lo ? ctl.t_start : lo;
        const double b = ctl.t_end < hi ? ctl.t_end : hi;
        rem = b - a;
        load_forcing2<ARITH>(d, p, c, r, l, Gm, L, sbc[g]);
        __builtin_amdgcn_wave_barrier();
        continue;
      }
    }
    bool pause = false;
    if (!finish) {
      if (attempts >= ctl.max_attempts) {
        dg.status = 2;
        if (l == 0) atomicOr(errflag, 2);
        finish = true;
      } else if (ctl.window > 0 && wn >= ctl.window) {
        pause = true;
      }
    }
    if (!finish && !pause) {
      ++attempts;
      ++wn;
      const bool clipped = !(dt < rem);
      const double h = clipped ? rem : dt;
      double f0[2][NV], c1[2][NV];
      double s0C[2], s0N[2], s1C[2], s1N[2];
      column_rhs2<ARITH>(p, L, bc, x, s0C, s0N, [&](int s, int n, double rr, double Fv) {
        f0[s][n] = rr;
        if (l == 0 && s == 0) F[0][n] = Fv;
      });
      const double p1 = psolve2<LPC, false>(x, f0, x, h, act, zs, dg.newton);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const double y = x[s][n] + (h * p1) * f0[s][n];
          c1[s][n] = y < 0.0 ? 0.0 : y;
        }
      column_rhs2<ARITH>(p, L, bc, c1, s1C, s1N, [&](int s, int n, double rr, double Fv) {
        f0[s][n] = (f0[s][n] + rr) * 0.5;
        if (l == 0 && s == 0) F[1][n] = Fv;
      });
      const double p2 = psolve2<LPC, true>(x, f0, c1, h, act, zs, dg.newton);
      double el[2];
      bool bad = false;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        double bn = 0.0, bd = 1.0;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const double y = x[s][n] + (h * p2) * f0[s][n];
          const double yp = y < 0.0 ? 0.0 : y;
          const double sc = p.emp_atol + p.emp_rtol * (yp > x[s][n] ? yp : x[s][n]);
          const double dv = fabs(yp - c1[s][n]);
          bad |= act[s] && ((dv != dv) || (sc != sc));
          if (dv * bd > bn * sc) {
            bn = dv;
            bd = sc;
          }
        }
        el[s] = bn / bd;
        bad |= act[s] && (el[s] != el[s]);
        if (!act[s]) el[s] = 0.0;
      }
      // the first tree level (lower layer first), then the lane butterfly
      const double elp = (el[1] > el[0] || el[1] != el[1]) ? el[1] : el[0];
      const double err = lg_max<LPC>(elp);
      if (group_any<LPC>(bad)) {
        dg.status = 1;
        if (l == 0) atomicOr(errflag, 1);
        finish = true;
      } else {
        const bool accept = (err <= 1.0) || !(h > p.emp_dt_min);
        double fac = err > 0.0 ? 0.9 * drsqrt(err) : 5.0;
        if (fac < 0.2) fac = 0.2;
        if (fac > 5.0) fac = 5.0;
        if (p1 < dg.p_min) dg.p_min = p1;
        if (p2 < dg.p_min) dg.p_min = p2;
        if (accept) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int n = 0; n < NV; ++n) {
              double y = x[s][n] + (h * p2) * f0[s][n];
              if (y < 0.0) {
                if (elem(n) >= 0 && act[s])
                  kadd(d.cellacc[(2 + elem(n)) * d.ncell + cell[s]], d.cellacc[(7 + elem(n)) * d.ncell + cell[s]],
                       0.0 - y);
                y = 0.0;
              }
              x[s][n] = y;
            }
          if (own) {
            kadd(fint, fintc, (h * p2) * ((F[0][l] + F[1][l]) * 0.5));
            flast = F[1][l];
          }
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            kadd(scell[0][s][threadIdx.x], scell[2][s][threadIdx.x], (h * p2) * ((s0C[s] + s1C[s]) * 0.5));
            kadd(scell[1][s][threadIdx.x], scell[3][s][threadIdx.x], (h * p2) * ((s0N[s] + s1N[s]) * 0.5));
          }
          rem = rem - h;
          dg.accepted += 1;
          if (err > 1.0) dg.forced += 1;
          dg.dt_last = h;
          if (h < dg.dt_minacc) dg.dt_minacc = h;
          const double prop = h * fac;
          dt = (clipped && dt > prop) ? dt : prop;
        } else {
          dg.rejected += 1;
          dt = h * fac;
        }
        if (dt < p.emp_dt_min) dt = p.emp_dt_min;
        if (dt > p.emp_dt_max) dt = p.emp_dt_max;
      }
    }
    if (finish || pause) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (act[s]) {
#pragma unroll
          for (int n = 0; n < NV; ++n) d.conc[n * d.ncell + cell[s]] = x[s][n];
          d.cellacc[cell[s]] = scell[0][s][threadIdx.x];
          d.cellacc[d.ncell + cell[s]] = scell[1][s][threadIdx.x];
          d.cellacc[5 * d.ncell + cell[s]] = scell[2][s][threadIdx.x];
          d.cellacc[6 * d.ncell + cell[s]] = scell[3][s][threadIdx.x];
        }
      }
      if (own) {
        d.colacc[(long long)l * d.ncol + c] = fint;
        d.colacc[(long long)(NV + l) * d.ncol + c] = fintc;
        d.flux[(long long)l * d.ncol + c] = flast;
      }
      const double zsum = lg_sum<LPC>((double)zs);
      if (l == 0) {
        dg.zero_sink += (int64_t)zsum;
        dg.dt_next = dt;
        d.diag[c] = dg;
        work[c] = attempts < 0x7fffffffll ? (int)attempts : 0x7fffffff;
        d.wrec[c] = pause ? r : r1 + 1;
        d.wrem[c] = rem;
        d.watt[c] = attempts;
        if (pause) atomicAdd(pending, 1);
      }
      have = false;
    }
  }
}

// ---------------------------------------------------------------------------
// linearly implicit adaptive stepper (method 7): ROS2 as a W-method
// ---------------------------------------------------------------------------
//
//   W k1 = f(c),  W k2 = f(c + h k1) - 2 k1,  c+ = c + h (3/2 k1 + 1/2 k2),
//   error estimate h (k1 + k2)/2 against the first-order c + h k1,
// gamma = 1 + 1/sqrt(2) (Verwer, Spee, Blom and Hundsdorfer 1999).  W is
// the product of the per-species tridiagonal transport factor
// B = I - gamma h J_T (Thomas sweeps, one lane per species, through LDS)
// and the per-cell reaction factor A = I - gamma h J_R (block solve in the
// lane's registers), plus one correction with the full matrix:
//   k0 = A^-1 B^-1 r,  k = k0 + A^-1 B^-1 (r - (I - gamma h (J_T + J_R)) k0).
// The transport coefficients come from the same diffusivities as the
// right-hand side, whose arithmetic form (reference or fast) is the
// instance's.  Budgets: top fluxes integrate as h/2 [(F0 + F1) + g (T1 +
// T2)] with T the linearised Dirichlet top-flux terms of the two solves,
// the DIC and N2 sinks as h/2 [(s0 + s1) + g grad s . (k1 + k2)]: exactly
// what the update moves.  Positivity: a new state below -1e-3 atol
// rejects the step (zero_sink counts these); smaller negative values are
// clamped to 0 and booked as clamp mass.  Failed local solves (a pivot
// that is not positive) reject the step with a quarter step (newton counts
// these).  Same operation sequence as the oracle's col_ros2_adaptive.

constexpr double ROS_GAMMA = 1.7071067811865475;

// two doubles in one 16-byte LDS access
typedef double dbl2 __attribute__((ext_vector_type(2)));

// per-group LDS of the stepper
template <int LPC>
struct alignas(16) RosShared {
  // Species rows padded by two doubles: the sweep of species n runs in lane
  // n, so the lanes read one pair of layers of 11 different rows at once;
  // with this pitch the 16-byte reads fall into different LDS banks
  double T[NV][LPC + 2];  // right-hand sides and solutions of the species sweeps
  // The transport factor is the same for all particulate variables ([0]) and
  // for all dissolved ones ([1]): they share diffusivity and top condition
  dbl2 BC[2][LPC];     // diagonal and super-diagonal coupling
  dbl2 AI[2][LPC];     // sub-diagonal coupling of the forward sweep, reciprocal pivot
  double E[2][LPC + 2];   // super-diagonal coupling times reciprocal pivot (back substitution)
  double top[2][NV];      // linearised Dirichlet top-flux terms of the two stages
};

// the lane's transport coefficients: D/dzc (D/dz at the top) of the
// particulate and dissolved variables, 1/(phi dz)
struct RosLane {
  double Gp, Gd, W;
};

// Matrix rows of both classes, one layer per lane: everything of the Thomas
// factorisation that is not on its serial chain.  Lanes beyond the column
// write identity rows.
template <int LPC>
__device__ __forceinline__ void ros_rows(RosShared<LPC> &R, const RosLane &C, int l, int K, bool act, double phi,
                                         double g, unsigned dirmask)
{
  const bool first = l == 0, last = l == K - 1;
  const double phu = lg_up(phi), phd = lg_dn(phi);
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const double G = m == 0 ? C.Gp : C.Gd;
    const double Gdn = lg_dn(G);
    const bool dir = (dirmask >> (m == 0 ? 0 : 5)) & 1u;
    const double s = ((!first || dir) ? G : 0.0) + (last ? 0.0 : Gdn);
    const double b = 1.0 + g * (C.W * (m == 0 ? s * phi : s));
    const double a = g * (m == 0 ? (C.W * G) * phu : C.W * G);
    const double c = g * (m == 0 ? (C.W * Gdn) * phd : C.W * Gdn);
    R.BC[m][l] = dbl2{act ? b : 1.0, act && !last ? c : 0.0};
    R.AI[m][l].x = act && !first ? a : 0.0;
  }
}

// The sweeps exist twice.  ros_*_lds (lane n < NV sweeps species n, all
// operands in LDS, IEEE divisions) serves columns of up to 16 layers and any
// value.  For LPC = 32 and 64 RosSweep does the same operations with the
// factor in registers: LDS traffic bounds the LDS form, because an access by
// 11 lanes costs a full wave's (68 cycles a layer against a chain of 24).
// A factor with its first sweep went from 6700 to 3300 cycles (24 layers), a
// sweep down from 2200 to 930 and up from 2700 to 850; a day of 3000
// columns of 20 to 40 layers, a spin-up's two chunks, from 445 to 243 ms.

// Thomas factor of species l's class and forward sweep of the first solve
template <int LPC>
__device__ __forceinline__ void ros_factor_lds(RosShared<LPC> &R, int l, int K)
{
  if (l < NV) {
    const int m = part(l) ? 0 : 1;
    double *T = R.T[l];
    const bool keep = l == 0 || l == 5;  // one lane per class stores the factor
    double e = 0.0, d = 0.0;
    for (int k = 0; k < K; ++k) {
      const dbl2 bc = R.BC[m][k];
      const double a = R.AI[m][k].x;
      const double piv = bc.x - a * e;  // a = 0 in the first row
      const double iv = 1.0 / piv;
      e = bc.y * iv;
      d = k > 0 ? (T[k] + a * d) * iv : T[k] * iv;
      T[k] = d;
      if (keep) {
        R.AI[m][k].y = iv;
        R.E[m][k] = e;
      }
    }
  }
}

// forward sweep of species l: T_k <- (T_k + a_k T_{k-1}) / pivot_k
template <int LPC>
__device__ __forceinline__ void ros_forward_lds(RosShared<LPC> &R, int l, int K)
{
  if (l < NV) {
    double *T = R.T[l];
    const dbl2 *AI = R.AI[part(l) ? 0 : 1];
    double d = T[0] * AI[0].y;
    T[0] = d;
    for (int k = 1; k < K; ++k) {
      d = (T[k] + AI[k].x * d) * AI[k].y;
      T[k] = d;
    }
  }
}

// back substitution of species l: T_k <- T_k + E_k T_{k+1}
template <int LPC>
__device__ __forceinline__ void ros_backward_lds(RosShared<LPC> &R, int l, int K)
{
  if (l < NV) {
    double *T = R.T[l];
    const double *E = R.E[part(l) ? 0 : 1];
    double d = T[K - 1];
    for (int k = K - 2; k >= 0; --k) {
      d = T[k] + E[k] * d;
      T[k] = d;
    }
  }
}

// value of lane J of the lane's row of 16
template <int J>
__device__ __forceinline__ double row_bcast(double v)
{
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + J, 0xf, 0xf, true));
}

// Sweeps of a column of more than 16 layers: the particulate species in
// lanes 0..5 of the group's first row of 16 lanes, the dissolved ones in
// lanes 0..4 of the second.  Lane j of a row keeps the rows j, j + 16, ... of
// its class's factor, and each step takes its coefficients by a row
// broadcast, one VALU move each.  A species' right-hand side is read from
// LDS once, swept down and up in registers and written back.  Layers beyond
// the column are identity rows with right-hand side 0, so a finite last value
// leaves T_{K-1} as it is; solve() leaves a column whose last value is not
// finite to the LDS form.
template <int LPC>
struct RosSweep {
  static constexpr int R16 = LPC / 16;
  double a[R16], iv[R16], E[R16];
  double *T;   // the lane's species row
  int m, j;    // class and lane of its row
  bool own;    // sweeps a species (the others run along)

  __device__ __forceinline__ void init(RosShared<LPC> &R, int l)
  {
    m = (l >> 4) & 1;
    j = l & 15;
    own = l < 32 && j < (m == 0 ? 6 : 5);
    T = R.T[m == 0 ? (j < 5 ? j : 10) : (j < 5 ? 5 + j : 5)];
  }
  // the factor from LDS: one that the LDS form made has the rows of the column
  // only, the rest are identity rows
  __device__ __forceinline__ void load_factor(const RosShared<LPC> &R, int K)
  {
#pragma unroll
    for (int i = 0; i < R16; ++i) {
      const dbl2 ai = R.AI[m][16 * i + j];
      const double e = R.E[m][16 * i + j];
      const bool in = 16 * i + j < K;
      a[i] = ai.x;
      iv[i] = in ? ai.y : 1.0;
      E[i] = in ? e : 0.0;
    }
  }
  template <int B>
  __device__ __forceinline__ void load_block(double (&t)[LPC]) const
  {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const dbl2 v = *reinterpret_cast<const dbl2 *>(T + 8 * B + 2 * q);
      t[8 * B + 2 * q] = v.x;
      t[8 * B + 2 * q + 1] = v.y;
    }
  }
  template <int B>
  __device__ __forceinline__ void store_block(const double (&t)[LPC])
  {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<dbl2 *>(T + 8 * B + 2 * q) = dbl2{t[8 * B + 2 * q], t[8 * B + 2 * q + 1]};
  }
  template <int B, int Q = 0>
  __device__ __forceinline__ void fwd_block(double (&t)[LPC], double &d) const
  {
    if constexpr (Q < 8) {
      constexpr int k = 8 * B + Q;
      d = (t[k] + row_bcast<k % 16>(a[k / 16]) * d) * row_bcast<k % 16>(iv[k / 16]);
      t[k] = d;
      fwd_block<B, Q + 1>(t, d);
    }
  }
  template <int B, int Q = 7>
  __device__ __forceinline__ void bwd_block(double (&t)[LPC], double &d) const
  {
    if constexpr (Q >= 0) {
      constexpr int k = 8 * B + Q;
      d = t[k] + row_bcast<k % 16>(E[k / 16]) * d;
      t[k] = d;
      bwd_block<B, Q - 1>(t, d);
    }
  }
  // factor and forward sweep together: the factor's chain is a
  // multiply-subtract, a reciprocal and a multiply per layer; every lane of
  // the row computes it, and lane k % 16 keeps row k
  template <int B, int Q = 0>
  __device__ __forceinline__ void fac_block(const double (&b)[R16], const double (&c)[R16], double (&t)[LPC],
                                            double &d, double &e)
  {
    if constexpr (Q < 8) {
      constexpr int k = 8 * B + Q;
      const double ak = row_bcast<k % 16>(a[k / 16]);
      const double piv = row_bcast<k % 16>(b[k / 16]) - ak * e;
      const double ivk = rcp_exact(piv);
      e = row_bcast<k % 16>(c[k / 16]) * ivk;
      d = (t[k] + ak * d) * ivk;
      t[k] = d;
      const bool mine = j == k % 16;
      iv[k / 16] = mine ? ivk : iv[k / 16];
      E[k / 16] = mine ? e : E[k / 16];
      fac_block<B, Q + 1>(b, c, t, d, e);
    }
  }
  template <int B = 0>
  __device__ __forceinline__ void load_all(double (&t)[LPC], int kw) const
  {
    if constexpr (B < LPC / 8) {
      if (8 * B < kw) {
        load_block<B>(t);
        load_all<B + 1>(t, kw);
      }
    }
  }
  template <int B = 0>
  __device__ __forceinline__ void store_all(const double (&t)[LPC], int kw)
  {
    if constexpr (B < LPC / 8) {
      if (8 * B < kw) {
        if (own) store_block<B>(t);
        store_all<B + 1>(t, kw);
      }
    }
  }
  template <int B = 0>
  __device__ __forceinline__ void forward(double (&t)[LPC], double &d, int kw) const
  {
    if constexpr (B < LPC / 8) {
      if (8 * B < kw) {
        fwd_block<B>(t, d);
        forward<B + 1>(t, d, kw);
      }
    }
  }
  template <int B = 0>
  __device__ __forceinline__ void factor(const double (&b)[R16], const double (&c)[R16], double (&t)[LPC], double &d,
                                         double &e, int kw)
  {
    if constexpr (B < LPC / 8) {
      if (8 * B < kw) {
        fac_block<B>(b, c, t, d, e);
        factor<B + 1>(b, c, t, d, e, kw);
      }
    }
  }
  template <int B = LPC / 8 - 1>
  __device__ __forceinline__ void backward(double (&t)[LPC], double &d, int kw) const
  {
    if constexpr (B >= 0) {
      if (8 * B < kw) bwd_block<B>(t, d);
      backward<B - 1>(t, d, kw);
    }
  }

  // a factor made in registers to where the LDS form reads it
  __device__ __forceinline__ void store_factor(RosShared<LPC> &R) const
  {
#pragma unroll
    for (int i = 0; i < R16; ++i) {
      R.AI[m][16 * i + j].y = iv[i];
      R.E[m][16 * i + j] = E[i];
    }
  }

  // B z = T for the group's species; FACTOR makes the factor first.  False
  // (with T untouched) when a pivot of the group is outside the range of
  // rcp_exact or a value is not finite: the LDS form then takes over, for this
  // group alone, so that a column does not depend on its neighbour in the wave.
  // At 64 lanes the later solves read the factor from LDS again: 12 doubles less
  // are live in between (3000 columns of 40 to 63 layers, reference form, 43
  // minutes: 208 -> 177 ms, fast form 168 -> 156 ms).
  template <bool FACTOR>
  __device__ __forceinline__ bool solve(RosShared<LPC> &R, int kw, int K)
  {
    if constexpr (!FACTOR && LPC == 64) load_factor(R, K);
    double t[LPC];
    double d = -0.0;  // a = 0 in the first row: x + 0 * -0 is x
    bool ok = true;
    load_all(t, kw);
    if (FACTOR) {
      double b[R16], c[R16], e = 0.0;
#pragma unroll
      for (int i = 0; i < R16; ++i) {
        const dbl2 bc = R.BC[m][16 * i + j];
        b[i] = bc.x;
        c[i] = bc.y;
        a[i] = R.AI[m][16 * i + j].x;
        iv[i] = 1.0;
        E[i] = 0.0;
      }
      factor(b, c, t, d, e, kw);
#pragma unroll
      for (int i = 0; i < R16; ++i) ok = ok && iv[i] > 0x1p-900 && iv[i] < 0x1p900;
    } else {
      forward(t, d, kw);
    }
    const bool good = !group_any<LPC>(!(ok && fabs(d) < INFINITY));
    if (good) {
      if (FACTOR) store_factor(R);
      backward(t, d, kw);
      store_all(t, kw);
    }
    return good;
  }
};

// the most layers of the wave's columns, in a scalar register (a group that
// has no column counts with its last one, which costs time only)
template <int LPC>
__device__ __forceinline__ int wave_layers(int K)
{
  int kw = __builtin_amdgcn_readlane(K, 0);
  if (LPC == 32) {
    const int k2 = __builtin_amdgcn_readlane(K, 32);
    kw = k2 > kw ? k2 : kw;
  }
  return kw < LPC ? kw : LPC;
}

// B^-1 r for the lane's layer: stage through LDS, sweep, read back.  FACTOR
// makes the factor first (from the rows in LDS).  kw: the most layers of the
// wave's columns.
template <int LPC, bool FACTOR>
__device__ __forceinline__ void ros_bsolve(RosShared<LPC> &R, RosSweep<LPC> &S, int l, int K, int kw, bool act,
                                           const double (&r)[NV], double (&v)[NV])
{
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int n = 0; n < NV; ++n) R.T[n][l] = act ? r[n] : 0.0;
  __builtin_amdgcn_wave_barrier();
  bool done = false;
  if constexpr (LPC > 16) done = S.template solve<FACTOR>(R, kw, K);
  if (!done) {
    if (FACTOR) ros_factor_lds<LPC>(R, l, K);
    else ros_forward_lds<LPC>(R, l, K);
    __builtin_amdgcn_wave_barrier();
    ros_backward_lds<LPC>(R, l, K);
    if constexpr (LPC == 32 && FACTOR) {
      __builtin_amdgcn_wave_barrier();
      S.load_factor(R, K);
    }
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int n = 0; n < NV; ++n) v[n] = act ? R.T[n][l] : 0.0;
  __builtin_amdgcn_wave_barrier();
}

// k = W^-1 r (AMF and one correction); r is overwritten.  Lane 0 stores
// the stage's linearised Dirichlet top-flux terms in top[n].  Returns the
// lane's local solve status.
template <int LPC, bool FACTOR>
__device__ __forceinline__ bool ros_wsolve(RosShared<LPC> &R, RosSweep<LPC> &S, const KJac &J, const RosLane &C,
                                           int l, int K, int kw, bool act, double g, unsigned dirmask, double phi,
                                           double (&r)[NV], double (&k)[NV], double *top)
{
  const double Gn_p = lg_dn(C.Gp), Gn_d = lg_dn(C.Gd);  // used above the last layer only
  double a[NV];
  ros_bsolve<LPC, FACTOR>(R, S, l, K, kw, act, r, a);
  bool ok = kjac_solve(J, g, a, k);  // k = k0
  kjac_apply(J, k, a);               // a = J_R k0
  // residual (r - k0) + g (J_T k0 + J_R k0), into r
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const bool pt = part(n);
    const double q = pt ? phi : 1.0;
    const double zp = k[n] * q;
    const double zpn = lg_dn(zp);
    const double Gn = pt ? Gn_p : Gn_d;
    const double Fd = l < K - 1 ? -(Gn * (zpn - zp)) : 0.0;
    double Fu = lg_up(Fd);
    if (l == 0) Fu = ((dirmask >> n) & 1u) ? -((pt ? C.Gp : C.Gd) * zp) : 0.0;
    const double t = (Fu - Fd) * C.W;
    r[n] = (r[n] - k[n]) + g * (t + a[n]);
  }
  ros_bsolve<LPC, false>(R, S, l, K, kw, act, r, a);  // a = v2
  if (l == 0) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const bool pt = part(n);
      top[n] = ((dirmask >> n) & 1u) ? 0.0 - (((pt ? C.Gp : C.Gd) * (pt ? phi : 1.0)) * (k[n] + a[n])) : 0.0;
    }
  }
  ok = kjac_solve(J, g, a, r) && ok;  // r = kc
#pragma unroll
  for (int n = 0; n < NV; ++n) k[n] = k[n] + r[n];
  return ok || !act;
}

// one wave per SIMD: the stepper's live state (state, two stage vectors,
// the reaction Jacobian) exceeds the 256 registers of two waves; with one
// wave the overflow goes to the accumulation registers instead of scratch
#ifndef SEDCOL_ROS_MIN_WAVES
#define SEDCOL_ROS_MIN_WAVES 1
#endif

template <int LPC, int ARITH, int BLK>
__global__ __launch_bounds__(BLK, SEDCOL_ROS_MIN_WAVES) void k_ros_adaptive(
    const Dev *dptr, const int *list, int nlist, const sedcol_params *__restrict__ pptr,
    const EmpCtl *__restrict__ cptr, int *next, int *pending, int *work, int *errflag)
{
  const Dev &d = *dptr;
  const sedcol_params &p = *pptr;
  const EmpCtl &ctl = *cptr;
  constexpr int G = BLK / LPC;
  __shared__ double sbc[G][2 * NV];
  __shared__ double sF[G][2][NV];
  __shared__ int sslot[G];
  __shared__ RosShared<LPC> sR[G];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const bool own = l < NV;
  double(*F)[NV] = sF[g];
  double bc[NV];
  auto boundary = [&]() {
    __builtin_amdgcn_wave_barrier();
    take_top(p, sbc[g], bc);
  };
  RosShared<LPC> &R = sR[g];
  const int r1 = ctl.r1;
  const unsigned dirmask = (p.bcup_part == 2 ? 0x41Fu : 0u) | (p.bcup_dis == 2 ? 0x3E0u : 0u);
  const double negtol = 1.0e-3 * p.emp_atol;

  int c = 0, r = 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  double x[NV];
  __shared__ double sacc[7][BLK];
  double &sinkC = sacc[0][threadIdx.x], &sinkN = sacc[1][threadIdx.x], &fint = sacc[2][threadIdx.x];
  double &sinkCc = sacc[3][threadIdx.x], &sinkNc = sacc[4][threadIdx.x], &fintc = sacc[5][threadIdx.x];
  double &flast = sacc[6][threadIdx.x];
  sedcol_coldiag dg;
  long long attempts = 0;
  int wn = 0;
  double dt = 0.0, rem = 0.0;
  bool have = false, act = false;

  RosLane C{0.0, 0.0, 0.0};
  RosSweep<LPC> S;
  S.init(R, l);
  auto coefficients = [&]() {
    // W-matrix coefficients of the record (the right-hand side's
    // diffusivities)
    if (ARITH == ARITH_FAST) {
      C = RosLane{L.Gb, L.Gd, L.W};
    } else {
      C = RosLane{L.Dbio / L.dzc, L.Ddis / L.dzc, 1.0 / (L.phi * L.dz)};
    }
    __builtin_amdgcn_wave_barrier();
  };

  for (;;) {
    if (!have) {
      if (l == 0) sslot[g] = atomicAdd(next, 1);
      __builtin_amdgcn_wave_barrier();
      const int s = sslot[g];
      __builtin_amdgcn_wave_barrier();
      if (s >= nlist) break;
      c = list[s];
      if (ctl.resume) {
        r = d.wrec[c];
        if (r > r1) continue;
        rem = d.wrem[c];
        attempts = d.watt[c];
      } else {
        r = ctl.r0 - 1;
        rem = 0.0;
        attempts = 0;
      }
      setup_lane(d, c, l, L, Gm, cell);
      act = L.active;
#pragma unroll
      for (int n = 0; n < NV; ++n) x[n] = act ? d.conc[n * d.ncell + cell] : 0.0;
      sinkC = act ? d.cellacc[cell] : 0.0;
      sinkN = act ? d.cellacc[d.ncell + cell] : 0.0;
      sinkCc = act ? d.cellacc[5 * d.ncell + cell] : 0.0;
      sinkNc = act ? d.cellacc[6 * d.ncell + cell] : 0.0;
      fint = own ? d.colacc[(long long)l * d.ncol + c] : 0.0;
      fintc = own ? d.colacc[(long long)(NV + l) * d.ncol + c] : 0.0;
      flast = own ? d.flux[(long long)l * d.ncol + c] : 0.0;
      dg = d.diag[c];
      dt = dg.dt_next;
      if (!(dt > 0.0)) dt = p.emp_dt_max;
      wn = 0;
      have = true;
      if (rem > 0.0) {
        load_forcing<LPC, ARITH>(d, p, c, r, Gm, L, sbc[g]);
        boundary();
        coefficients();
      }
    }
    bool finish = false;
    if (!(rem > 0.0)) {
      ++r;
      if (r > r1) {
        finish = true;
      } else {
        const double lo = (r == 0) ? -INFINITY : d.t0 + (double)r * d.dt_rec;
        const double hi = (r == d.nrec - 1) ? INFINITY : d.t0 + (double)(r + 1) * d.dt_rec;
        const double a = ctl.t_start > lo ? ctl.t_start : lo;
        const double b = ctl.t_end < hi ? ctl.t_end : hi;
        rem = b - a;
        load_forcing<LPC, ARITH>(d, p, c, r, Gm, L, sbc[g]);
        boundary();
        coefficients();
        continue;
      }
    }
    bool pause = false;
    if (!finish) {
      if (attempts >= ctl.max_attempts) {
        dg.status = 2;
        if (l == 0) atomicOr(errflag, 2);
        finish = true;
      } else if (ctl.window > 0 && wn >= ctl.window) {
        pause = true;
      }
    }
    if (!finish && !pause) {
      ++attempts;
      ++wn;
      const bool clipped = !(dt < rem);
      const double h = clipped ? rem : dt;
      const double gh = ROS_GAMMA * h;
      const int K = L.K;
      const int kw = wave_layers<LPC>(K);
      double f[NV], k1[NV], k2[NV];
      double s0C, s0N, s1C = 0.0, s1N = 0.0;
      double Ft[NV];
      column_rhs<LPC, ARITH, 0>(p, L, bc, x, s0C, s0N, [&](int n, double rr, double Fv) {
        f[n] = rr;
        Ft[n] = Fv;
      });
      store_top(l == 0, Ft, F[0]);
      ros_rows<LPC>(R, C, l, K, act, L.phi, gh, dirmask);
      // The Jacobian stays live for the second stage, and with it the local
      // solves' pivots: a spin-up of 3000 columns (fast form) takes 165 ms against
      // 171 with a second evaluation, though 64 lanes then have 172 to 220 bytes
      // of scratch.
      KJac J;
      kin_jac(p, L.fT, x, J);
      bool ok = ros_wsolve<LPC, true>(R, S, J, C, l, K, kw, act, gh, dirmask, L.phi, f, k1, R.top[0]);
      double gC = kjac_sinkC(J, k1);
      double gN = kjac_sinkN(J, k1);
      bool fail = group_any<LPC>(!ok);
      if (!fail) {
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const double y = x[n] + h * k1[n];
          f[n] = y < 0.0 ? 0.0 : y;
        }
        double c1[NV];
#pragma unroll
        for (int n = 0; n < NV; ++n) c1[n] = f[n];
        column_rhs<LPC, ARITH, 0>(p, L, bc, c1, s1C, s1N, [&](int n, double rr, double Fv) {
          f[n] = rr - 2.0 * k1[n];
          Ft[n] = Fv;
        });
        store_top(l == 0, Ft, F[1]);
        ok = ros_wsolve<LPC, false>(R, S, J, C, l, K, kw, act, gh, dirmask, L.phi, f, k2, R.top[1]);
        fail = group_any<LPC>(!ok);
        gC = gC + kjac_sinkC(J, k2);
        gN = gN + kjac_sinkN(J, k2);
      }
      double bn = 0.0, bd = 1.0;
      bool bad = false, neg = false;
      if (!fail) {
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const double y = x[n] + h * (1.5 * k1[n] + 0.5 * k2[n]);
          const double yp = y < 0.0 ? 0.0 : y;
          const double sc = p.emp_atol + p.emp_rtol * (yp > x[n] ? yp : x[n]);
          const double dv = fabs(h * (0.5 * k1[n] + 0.5 * k2[n]));
          bad |= (dv != dv) || (sc != sc);
          neg |= y < 0.0 - negtol;
          if (dv * bd > bn * sc) {
            bn = dv;
            bd = sc;
          }
        }
      }
      double el = bn / bd;
      bad |= el != el;
      if (!act) {
        el = 0.0;
        bad = false;
        neg = false;
      }
      const double err = lg_max<LPC>(el);
      neg = group_any<LPC>(neg);
      if (group_any<LPC>(bad) || (fail && !(h > p.emp_dt_min))) {
        dg.status = 1;
        if (l == 0) atomicOr(errflag, 1);
        finish = true;
      } else {
        const bool accept = !fail && ((err <= 1.0 && !neg) || !(h > p.emp_dt_min));
        double fac = err > 0.0 ? 0.9 * drsqrt(err) : 5.0;
        if (fac < 0.2) fac = 0.2;
        if (fac > 5.0) fac = 5.0;
        if (accept) {
          bool odd = false;
#pragma unroll
          for (int n = 0; n < NV; ++n) {
            x[n] = x[n] + h * (1.5 * k1[n] + 0.5 * k2[n]);
            odd |= x[n] < 0.0;
          }
          if (__any(odd)) {
#pragma unroll
            for (int n = 0; n < NV; ++n)
              if (x[n] < 0.0) {
                if (elem(n) >= 0 && act)
                  kadd(d.cellacc[(2 + elem(n)) * d.ncell + cell], d.cellacc[(7 + elem(n)) * d.ncell + cell],
                       0.0 - x[n]);
                x[n] = 0.0;
              }
          }
          __builtin_amdgcn_wave_barrier();
          if (own) {
            kadd(fint, fintc, (h * 0.5) * ((F[0][l] + F[1][l]) + gh * (R.top[0][l] + R.top[1][l])));
            flast = F[1][l];
          }
          __builtin_amdgcn_wave_barrier();
          kadd(sinkC, sinkCc, (h * 0.5) * ((s0C + s1C) + gh * gC));
          kadd(sinkN, sinkNc, (h * 0.5) * ((s0N + s1N) + gh * gN));
          rem = rem - h;
          dg.accepted += 1;
          if (err > 1.0 || neg) dg.forced += 1;
          dg.dt_last = h;
          if (h < dg.dt_minacc) dg.dt_minacc = h;
          const double prop = h * fac;
          dt = (clipped && dt > prop) ? dt : prop;
        } else {
          dg.rejected += 1;
          if (fail) {
            dg.newton += 1;
            dt = h * 0.25;
          } else if (err <= 1.0) {
            dg.zero_sink += 1;
            dt = h * 0.5;
          } else {
            dt = h * fac;
          }
        }
        if (dt < p.emp_dt_min) dt = p.emp_dt_min;
        if (dt > p.emp_dt_max) dt = p.emp_dt_max;
      }
    }
    if (finish || pause) {
#pragma unroll
      for (int n = 0; n < NV; ++n)
        if (act) d.conc[n * d.ncell + cell] = x[n];
      if (act) {
        d.cellacc[cell] = sinkC;
        d.cellacc[d.ncell + cell] = sinkN;
        d.cellacc[5 * d.ncell + cell] = sinkCc;
        d.cellacc[6 * d.ncell + cell] = sinkNc;
      }
      if (own) {
        d.colacc[(long long)l * d.ncol + c] = fint;
        d.colacc[(long long)(NV + l) * d.ncol + c] = fintc;
        d.flux[(long long)l * d.ncol + c] = flast;
      }
      if (l == 0) {
        dg.dt_next = dt;
        d.diag[c] = dg;
        work[c] = attempts < 0x7fffffffll ? (int)attempts : 0x7fffffff;
        d.wrec[c] = pause ? r : r1 + 1;
        d.wrem[c] = rem;
        d.watt[c] = attempts;
        if (pause) atomicAdd(pending, 1);
      }
      have = false;
    }
  }
}

// ---------------------------------------------------------------------------
// ADAPTIVE_EULER (solver_library.F90:104-140): the reject rule is global, so
// each sub-step is a right-hand side, a domain-wide check and a commit
// ---------------------------------------------------------------------------

// Per attempt: the right-hand side with the relative-change test (k_ae_rhs; or
// the test alone, k_ae_check, when the step was quartered and the rates are
// still those of the state), then k_ae_commit, which looks at the vote and
// leaves the state alone if the step has to be quartered.  The host reads the
// vote behind the commit and does the same comparison, so a step that is not
// quartered costs two launches and one wait (four launches, a memset and a
// wait between them before).  The votes alternate between two flags: a commit
// clears the next attempt's.
__device__ __forceinline__ bool ae_violates(double x, double r, double dt_red, double rcm)
{
  const double c1 = x + dt_red * r;
  return (c1 - (1.0 + rcm) * x) < 0.0;
}

template <int LPC, int ARITH>
__global__ __launch_bounds__(BLOCK) void k_ae_rhs(Dev d, const int *list, int nlist, sedcol_params p, int rec,
                                                  double dt_red, double *r_out, double *s_out, int *viol)
{
  constexpr int G = BLOCK / LPC;
  __shared__ double sbc[G][2 * NV];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  const bool valid = slot < nlist;
  const int c = valid ? list[slot] : 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  if (valid) {
    setup_lane(d, c, l, L, Gm, cell);
    load_forcing<LPC, ARITH>(d, p, c, rec, Gm, L, sbc[g]);
  }
  __syncthreads();
  if (!valid) return;
  double x[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) x[n] = L.active ? d.conc[n * d.ncell + cell] : 0.0;
  double sC, sN;
  bool v = false;
  const double rcm = p.relative_change_min;
  column_rhs<LPC, ARITH>(p, L, sbc[g], x, sC, sN, [&](int n, double r, double F) {
    if (L.active) r_out[n * d.ncell + cell] = r;
    if (l == 0) d.flux[(long long)n * d.ncol + c] = F;
    v |= L.active && ae_violates(x[n], r, dt_red, rcm);
  }, &d.zw);
  if (L.active) {
    s_out[cell] = sC;
    s_out[d.ncell + cell] = sN;
  }
  if (v) atomicOr(viol, 1);
}

template <int LPC>
__global__ __launch_bounds__(BLOCK) void k_ae_check(Dev d, const int *list, int nlist, double dt_red, double rcm,
                                                    const double *r_in, int *viol)
{
  constexpr int G = BLOCK / LPC;
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  if (slot >= nlist) return;
  const int c = list[slot];
  const int o = d.off[c], K = d.off[c + 1] - o;
  if (l >= K) return;
  const long long cell = (long long)o + l;
  bool v = false;
#pragma unroll
  for (int n = 0; n < NV; ++n) v |= ae_violates(d.conc[n * d.ncell + cell], r_in[n * d.ncell + cell], dt_red, rcm);
  if (v) atomicOr(viol, 1);
}

// minimum clamp of one cell after an ode_solver call (fabm_sediment_component.F90:1726-1731):
// the clamped value; mass to the budget array
__device__ __forceinline__ double clamp_cell(const Dev &d, int n, long long cell, double x)
{
  if (x < 0.0) {
    if (elem(n) >= 0)
      kadd(d.cellacc[(2 + elem(n)) * d.ncell + cell], d.cellacc[(7 + elem(n)) * d.ncell + cell], 0.0 - x);
    x = 0.0;
  }
  return x;
}

// the step dt_red, unless the vote *viol asks for a smaller one and dt_red is
// above dt_min; clamp: also the minimum clamp and the NaN test (errflag bit 1)
// that follow a whole step; *clear (or null) is set to 0
template <int LPC>
__global__ __launch_bounds__(BLOCK) void k_ae_commit(Dev d, const int *list, int nlist, double dt_red, double dt_min,
                                                     int clamp, const double *r_in, const double *s_in,
                                                     const int *viol, int *clear, int *errflag)
{
  constexpr int G = BLOCK / LPC;
  if (clear && blockIdx.x == 0 && threadIdx.x == 0) *clear = 0;
  if (*viol && dt_red > dt_min) return;
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  if (slot >= nlist) return;
  const int c = list[slot];
  const int o = d.off[c], K = d.off[c + 1] - o;
  if (l < NV)
    kadd(d.colacc[(long long)l * d.ncol + c], d.colacc[(long long)(NV + l) * d.ncol + c],
         dt_red * d.flux[(long long)l * d.ncol + c]);
  if (l == 0) {
    sedcol_coldiag dg = d.diag[c];
    dg.accepted += 1;
    dg.dt_last = dt_red;
    if (dt_red < dg.dt_minacc) dg.dt_minacc = dt_red;
    d.diag[c] = dg;
  }
  if (l >= K) return;
  const long long cell = (long long)o + l;
  bool nan = false;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    double x = d.conc[n * d.ncell + cell] + dt_red * r_in[n * d.ncell + cell];
    if (clamp) {
      nan |= x != x;
      x = clamp_cell(d, n, cell, x);
    }
    d.conc[n * d.ncell + cell] = x;
  }
  kadd(d.cellacc[cell], d.cellacc[5 * d.ncell + cell], dt_red * s_in[cell]);
  kadd(d.cellacc[d.ncell + cell], d.cellacc[6 * d.ncell + cell], dt_red * s_in[d.ncell + cell]);
  if (nan) atomicOr(errflag, 1);
}

// ADAPTIVE_EULER steps of a small domain in one workgroup: every wet column
// of the list is a lane group of the block, so the reference's global rule
// (the step is quartered while any cell of the domain fails the
// relative-change test, solver_library.F90:100-140) is a block-wide vote
// instead of a flag read by the host.  Per attempt the same operations as
// k_ae_rhs and k_ae_commit, so the results are those of the multi-launch path bit for bit.  The state
// stays in registers; the top fluxes of the last right-hand side go to LDS
// for the lanes that accumulate them.  *min_dt receives the smallest step
// taken.  A launch stops after kAeFusedMaxAttempts attempts (errflag bit 2).
// The time is that of one dependent chain, so a domain of one wave runs as a
// block of one wave (BLK = 64): the vote and the barriers stay inside the
// wave and a lane has all the registers it asks for.
template <int LPC, int ARITH, int BLK>
__global__ __launch_bounds__(BLK) void k_ae_fused(const Dev *dptr, const int *list, int nlist,
                                                  const sedcol_params *__restrict__ pptr, int rec, double dt,
                                                  int nsteps, int *errflag, double *min_dt)
{
  // domain and parameters through pointers to device copies: passed by
  // value they would sit in scalar registers for the whole run and spill
  const Dev &d = *dptr;
  const sedcol_params &p = *pptr;
  constexpr int G = BLK / LPC;
  constexpr bool ONE = BLK == 64;  // one wave
  auto sync = [] {
    if constexpr (ONE) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
  };
  __shared__ double sbc[G][2 * NV];
  __shared__ double sF[G][NV];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const bool valid = g < nlist;
  const int c = valid ? list[g] : 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  if (valid) {
    setup_lane(d, c, l, L, Gm, cell);
    load_forcing<LPC, ARITH>(d, p, c, rec, Gm, L, sbc[g]);
  } else {
    L.l = l;
    L.K = 0;
    L.active = false;
  }
  __syncthreads();
  const bool act = valid && L.active;
  const bool own = valid && l < NV;
  // boundary values: in registers for one wave, as in k_fixed
  constexpr int TF = ONE ? 0 : NV;
  double rbc[NV];
  if constexpr (ONE) take_top(p, sbc[g], rbc);
  const double *bc = ONE ? rbc : sbc[g];
  // Two waves per SIMD (BLK = 512) have no registers for the rates between an
  // evaluation and its step: in LDS 12 to 252 bytes of scratch per lane are left
  // of 92 to 428, and four calls of 1800 s for 20 columns of 16 layers take 245 us
  // instead of 360 (fast form 207 for 241, extended form 403 for 762).
  constexpr bool RLDS = BLK > 256;
  __shared__ double srate[RLDS ? NV : 1][RLDS ? BLK : 1];
  double x[NV], rreg[NV];
  auto r = [&](int n) -> double & {
    if constexpr (RLDS) return srate[n][threadIdx.x];
    else return rreg[n];
  };
#pragma unroll
  for (int n = 0; n < NV; ++n) x[n] = act ? d.conc[n * d.ncell + cell] : 0.0;
  double sC = 0.0, sN = 0.0;
  // sums touched only by accepted attempts: in registers for one wave, else
  // in LDS, leaving the registers to the right-hand side.  The DIC and N2
  // sinks with their compensations, the lane's top-flux sum and compensation
  __shared__ double sacc[6][ONE ? 1 : BLK];
  double racc[6];
  const int t = threadIdx.x;
  auto acc = [&](int i) -> double & {
    if constexpr (ONE) return racc[i];
    else return sacc[i][t];
  };
  acc(0) = act ? d.cellacc[cell] : 0.0;
  acc(1) = act ? d.cellacc[d.ncell + cell] : 0.0;
  acc(2) = act ? d.cellacc[5 * d.ncell + cell] : 0.0;
  acc(3) = act ? d.cellacc[6 * d.ncell + cell] : 0.0;
  acc(4) = own ? d.colacc[(long long)l * d.ncol + c] : 0.0;
  acc(5) = own ? d.colacc[(long long)(NV + l) * d.ncol + c] : 0.0;
  // the attempts of this launch enter the columns' diagnostics at its end
  // (every column takes the same steps)
  int accepted = 0;
  double dt_last = 0.0;
  const double rcm = p.relative_change_min;
  double mind = INFINITY;
  int attempts = 0;
  bool stop = false;
  for (int s = 0; s < nsteps && !stop; ++s) {
    double dt_int = 0.0, dt_red = dt;
    bool need = true;
    while (dt_int < dt) {
      if (++attempts > kAeFusedMaxAttempts) {
        if (threadIdx.x == 0) atomicOr(errflag, 2);
        stop = true;
        break;
      }
      if (need) {
        if (valid) {
          double Ft[NV];
          column_rhs<LPC, ARITH, TF>(p, L, bc, x, sC, sN, [&](int n, double rr, double F) {
            r(n) = rr;
            Ft[n] = F;
          }, &d.zw);
          store_top(l == 0, Ft, sF[g]);
        }
        need = false;
        sync();
      }
      bool v = false;
      if (act) {
#pragma unroll
        for (int n = 0; n < NV; ++n) v |= ae_violates(x[n], r(n), dt_red, rcm);
      }
      const int viol = ONE ? __any(v) : __syncthreads_or(v);
      if (viol && dt_red > p.dt_min) {
        dt_red = dt_red * 0.25;  // the state is unchanged: the right-hand side is reused
      } else {
        if (dt_red < mind) mind = dt_red;
        if (own) kadd(acc(4), acc(5), dt_red * sF[g][l]);
        ++accepted;
        dt_last = dt_red;
        if (act) {
#pragma unroll
          for (int n = 0; n < NV; ++n) x[n] = x[n] + dt_red * r(n);
          kadd(acc(0), acc(2), dt_red * sC);
          kadd(acc(1), acc(3), dt_red * sN);
        }
        dt_int = dt_int + dt_red;
        need = true;
        // the lanes reading sF are done before the next evaluation writes it
        sync();
      }
    }
    if (stop) break;
    if (p.clamp && act) {
      bool odd = false;
#pragma unroll
      for (int n = 0; n < NV; ++n) odd |= !(x[n] >= 0.0);
      if (__any(odd)) {
        bool nan = false;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          nan |= x[n] != x[n];
          if (x[n] < 0.0) {
            if (elem(n) >= 0)
              kadd(d.cellacc[(2 + elem(n)) * d.ncell + cell], d.cellacc[(7 + elem(n)) * d.ncell + cell], 0.0 - x[n]);
            x[n] = 0.0;
          }
        }
        if (nan) atomicOr(errflag, 1);
      }
    }
  }
  if (act) {
#pragma unroll
    for (int n = 0; n < NV; ++n) d.conc[n * d.ncell + cell] = x[n];
    d.cellacc[cell] = acc(0);
    d.cellacc[d.ncell + cell] = acc(1);
    d.cellacc[5 * d.ncell + cell] = acc(2);
    d.cellacc[6 * d.ncell + cell] = acc(3);
  }
  if (own) {
    d.colacc[(long long)l * d.ncol + c] = acc(4);
    d.colacc[(long long)(NV + l) * d.ncol + c] = acc(5);
    if (attempts > 0) d.flux[(long long)l * d.ncol + c] = sF[g][l];
  }
  if (valid && l == 0 && accepted > 0) {
    sedcol_coldiag dg = d.diag[c];
    dg.accepted += accepted;
    dg.dt_last = dt_last;
    if (mind < dg.dt_minacc) dg.dt_minacc = mind;
    d.diag[c] = dg;
  }
  if (threadIdx.x == 0) *min_dt = mind;
}

// ---------------------------------------------------------------------------
// column reductions: budget, inventory, steady-state residual
// ---------------------------------------------------------------------------

template <int LPC>
__global__ __launch_bounds__(BLOCK) void k_budget(Dev d, const int *list, int nlist, double *budget)
{
  constexpr int G = BLOCK / LPC;
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  if (slot >= nlist) return;
  const int c = list[slot];
  const int o = d.off[c], K = d.off[c + 1] - o;
  const bool act = l < K;
  const long long cell = (long long)o + l;
  const double w = act ? d.phi[cell] * d.dz[cell] : 0.0;
  double *b = budget + (long long)c * SEDCOL_NBUD;
  if (l < NV) b[l] = d.colacc[(long long)l * d.ncol + c] + d.colacc[(long long)(NV + l) * d.ncol + c];
#pragma unroll
  for (int a = 0; a < 5; ++a) {
    const double v = act ? w * (d.cellacc[a * d.ncell + cell] + d.cellacc[(5 + a) * d.ncell + cell]) : 0.0;
    const double s = lg_sum<LPC>(v);
    if (l == 0) b[NV + a] = s;
  }
}

template <int LPC>
__global__ __launch_bounds__(BLOCK) void k_inventory(Dev d, const int *list, int nlist, double *inv)
{
  constexpr int G = BLOCK / LPC;
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  if (slot >= nlist) return;
  const int c = list[slot];
  const int o = d.off[c], K = d.off[c + 1] - o;
  const bool act = l < K;
  const long long cell = (long long)o + l;
  const double w = act ? d.phi[cell] * d.dz[cell] : 0.0;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const double v = act ? w * d.conc[n * d.ncell + cell] : 0.0;
    const double s = lg_sum<LPC>(v);
    if (l == 0) inv[(long long)n * d.ncol + c] = s;
  }
}

template <int LPC, int ARITH>
__global__ __launch_bounds__(BLOCK) void k_residual(Dev d, const int *list, int nlist, sedcol_params p, int rec,
                                                    const double *cfloor, double *resid, double *flux)
{
  constexpr int G = BLOCK / LPC;
  __shared__ double sbc[G][2 * NV];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  const bool valid = slot < nlist;
  const int c = valid ? list[slot] : 0;
  Lane L;
  Geo Gm;
  long long cell = 0;
  if (valid) {
    setup_lane(d, c, l, L, Gm, cell);
    load_forcing<LPC, ARITH>(d, p, c, rec, Gm, L, sbc[g]);
  }
  __syncthreads();
  if (!valid) return;
  double x[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) x[n] = L.active ? d.conc[n * d.ncell + cell] : 0.0;
  double sC, sN, m = 0.0;
  column_rhs<LPC, ARITH>(p, L, sbc[g], x, sC, sN, [&](int n, double r, double F) {
    const double ax = fabs(x[n]);
    const double den = ax > cfloor[n] ? ax : cfloor[n];
    const double e = fabs(r) / den;
    if (L.active && (e > m || e != e)) m = e;
    if (l == 0 && flux) flux[(long long)n * d.ncol + c] = F;
  }, &d.zw);
  m = lg_max<LPC>(m);
  if (l == 0) resid[c] = m;
}

// ---------------------------------------------------------------------------
// boundary conditions from the pelagic fields at the soil surface
// (get_boundary_conditions, fabm_sediment_component.F90:1865-2030): one
// thread per listed column, writing forcing record 0
// ---------------------------------------------------------------------------

__global__ void k_assemble(Dev d, const int *list, int nlist, double D0, int bcup_dis, unsigned present,
                           const double *ts, const double *cs, const double *ws, double *temp, double *cbw,
                           double *fup)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nlist) return;
  const int c = list[i];
  const long long top = d.off[c];
  if (ts) temp[c] = ts[c];  // :1903-1939
  for (int n = 0; n < NV; ++n) {
    if (!((present >> n) & 1u)) continue;  // field absent: left as it is (:1963-1967)
    const long long k = (long long)n * d.ncol + c;
    if (part(n)) {
      fup[k] = -(cs[k] * ws[k]);  // :1978-1986, downward positive
    } else {
      cbw[k] = cs[k];  // :1989-2000
      if (bcup_dis == 1) {
        // :2012-2014, in its operation order
        double x = (d.conc[n * d.ncell + top] - cbw[k]) / d.dz[top];
        x = x * ((d.biot[c] + D0) + temp[c] * 0.035);
        x = x * d.phi[top];
        x = x / 86400.0;
        x = x / 10000.0;
        fup[k] = -x;
      } else {
        fup[k] = 0.0;  // :2021
      }
    }
  }
}

void launch_assemble(hipStream_t st, const Dev &d, const int *list, int n, const sedcol_params &p, unsigned present,
                     const double *ts, const double *cs, const double *ws, double *temp, double *cbw, double *fup)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_assemble, dim3((n + 255) / 256), dim3(256), 0, st, d, list, n, p.D0, (int)p.bcup_dis, present,
                     ts, cs, ws, temp, cbw, fup);
}

// ---------------------------------------------------------------------------
// launch helpers (host)
// ---------------------------------------------------------------------------

template <int LPC>
static inline dim3 grid_for(int n)
{
  constexpr int G = BLOCK / LPC;
  return dim3((unsigned)((n + G - 1) / G));
}

// kernel instance for the parameters: the extended reference form for
// BcUp = 4 and bioturbation profile 3 (the host marks the latter with
// arith = ARITH_EXT), the fast form where it applies, else the reference form
static inline int arith_form(const sedcol_params &p)
{
  if (p.arith == ARITH_EXT || p.bcup_part == 4) return ARITH_EXT;
  if (p.arith == SEDCOL_ARITH_FAST && p.bcdown != 2) return ARITH_FAST;
  return ARITH_REF;
}

#define SC_DISPATCH_LPC(lpc, ...)                                \
  switch (lpc) {                                                 \
    case 16: { constexpr int LPC = 16; __VA_ARGS__; } break;     \
    case 32: { constexpr int LPC = 32; __VA_ARGS__; } break;     \
    default: { constexpr int LPC = 64; __VA_ARGS__; } break;     \
  }
#define SC_DISPATCH_ARITH(p, ...)                                          \
  switch (arith_form(p)) {                                                 \
    case ARITH_FAST: { constexpr int AR = ARITH_FAST; __VA_ARGS__; } break; \
    case ARITH_EXT: { constexpr int AR = ARITH_EXT; __VA_ARGS__; } break;   \
    default: { constexpr int AR = ARITH_REF; __VA_ARGS__; } break;          \
  }

void launch_rhs(int lpc, hipStream_t st, const Dev &d, const int *list, int n, const sedcol_params &p, int rec,
                const double *conc, double *rhs, double *flux, double *sinks)
{
  SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_rhs<LPC, AR>), grid_for<LPC>(n), dim3(BLOCK), 0,
                                                               st, d, list, n, p, rec, conc, rhs, flux, sinks)));
}

// lanes of one wave on each of the 1024 SIMDs
constexpr long long kSimdLanes = 1024 * 64;

void launch_fixed(int lpc, int method, hipStream_t st, const Dev &d, const int *list, int n,
                  const sedcol_params &p, int rec, double dt, int nsteps, int *errflag)
{
  const bool full = (long long)n * lpc > kSimdLanes;
#define SC_FIX(M, W)                                                                                             \
  SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, {                                                                      \
                      auto *k = k_fixed<LPC, M, AR, W, false>;                                                     \
                      if (full) k = k_fixed<LPC, M, AR, W, fixed_split(M, AR, W)>;                                 \
                      hipLaunchKernelGGL(k, grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n, p, rec, dt, nsteps,  \
                                         errflag);                                                                 \
                    }))
  const bool geo = p.emp_weights == 1;
  switch (method) {
    case SEDCOL_EULER: SC_FIX(SEDCOL_EULER, 0); break;
    case SEDCOL_RUNGE_KUTTA_4: SC_FIX(SEDCOL_RUNGE_KUTTA_4, 0); break;
    case SEDCOL_RUNGE_KUTTA_4_38: SC_FIX(SEDCOL_RUNGE_KUTTA_4_38, 0); break;
    case SEDCOL_EMP1:
      if (geo) {
        SC_FIX(SEDCOL_EMP1, 1);
      } else {
        SC_FIX(SEDCOL_EMP1, 0);
      }
      break;
    default:
      if (geo) {
        SC_FIX(SEDCOL_EMP2, 1);
      } else {
        SC_FIX(SEDCOL_EMP2, 0);
      }
      break;
  }
#undef SC_FIX
}

// blocks of a work-queue kernel that are resident at once on the current
// device, cached per device and kernel instance (threads that race on a
// first query store the same value).  PW = 2 selects the linearly implicit
// kernel k_ros_adaptive, PW = 3 k_emp_adaptive2 (two layers per lane),
// otherwise k_emp_adaptive with Patankar weights PW.
template <int LPC, int AR, int BLK, int PW>
static int emp_resident()
{
  constexpr int kMaxDev = 64;
  static std::atomic<int> cached[kMaxDev];  // static storage: starts at zero
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 1024;
  std::atomic<int> *slot = (dev >= 0 && dev < kMaxDev) ? &cached[dev] : nullptr;
  int v = slot ? slot->load(std::memory_order_relaxed) : 0;
  if (v > 0) return v;
  hipDeviceProp_t prop;
  int per_cu = 0;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 1024;
  hipError_t e;
  if constexpr (PW == 2)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_ros_adaptive<LPC, AR, BLK>, BLK, 0);
  else if constexpr (PW == 3)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_emp_adaptive2<LPC, AR, BLK>, BLK, 0);
  else
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_emp_adaptive<LPC, AR, BLK, PW>, BLK, 0);
  if (e != hipSuccess) per_cu = 1;
  v = (per_cu > 0 ? per_cu : 1) * prop.multiProcessorCount;
  if (slot) slot->store(v, std::memory_order_relaxed);
  return v;
}

#define SC_DISPATCH_BLK(blk, ...)                                \
  switch (blk) {                                                 \
    case 64: { constexpr int BLK = 64; __VA_ARGS__; } break;     \
    case 128: { constexpr int BLK = 128; __VA_ARGS__; } break;   \
    case 256: { constexpr int BLK = 256; __VA_ARGS__; } break;   \
    default: return false;                                       \
  }
#define SC_DISPATCH_PW(p, ...)                                   \
  switch ((p).emp_weights) {                                     \
    case 1: { constexpr int PW = 1; __VA_ARGS__; } break;        \
    default: { constexpr int PW = 0; __VA_ARGS__; } break;       \
  }

static bool emp_shape_ok(int lpc, int blk)
{
  return (lpc == 16 || lpc == 32 || lpc == 64) && (blk == 64 || blk == 128 || blk == 256);
}

// the linearly implicit kernel has the reference and fast forms only
#define SC_DISPATCH_ROS_ARITH(p, ...)                                          \
  switch (arith_form(p)) {                                                     \
    case ARITH_FAST: { constexpr int AR = ARITH_FAST; __VA_ARGS__; } break;     \
    case ARITH_REF: { constexpr int AR = ARITH_REF; __VA_ARGS__; } break;       \
    default: return false;                                                     \
  }

static bool ros_selected(const sedcol_params &p) { return p.adaptive_method == SEDCOL_ROS2_ADAPTIVE; }

bool emp2_supported(const sedcol_params &p)
{
  return !ros_selected(p) && p.emp_weights == 0 && arith_form(p) != ARITH_EXT;
}

int emp_resident_blocks(int lpc, int blk, int lpl, const sedcol_params &p)
{
  if (!emp_shape_ok(lpc, blk)) return 0;
  if (lpl == 2 && (lpc < 16 || !emp2_supported(p))) return 0;
  int out = 0;
  auto body = [&]() -> bool {
    if (lpl == 2) {
      SC_DISPATCH_ROS_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, out = emp_resident<LPC, AR, BLK, 3>())));
    } else if (ros_selected(p)) {
      SC_DISPATCH_ROS_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, out = emp_resident<LPC, AR, BLK, 2>())));
    } else {
      SC_DISPATCH_PW(p, SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, out = emp_resident<LPC, AR, BLK, PW>()))));
    }
    return true;
  };
  body();
  return out;
}

bool launch_emp_adaptive(int lpc, int blk, int lpl, hipStream_t st, const Dev *d_dev, const int *list, int n,
                         const sedcol_params &p, const sedcol_params *d_params, const EmpCtl *d_ctl, int *next,
                         int *pending, int *work, int *errflag)
{
  if (!emp_shape_ok(lpc, blk)) return false;
  if (lpl == 2) {
    if (lpc < 16 || !emp2_supported(p)) return false;
    SC_DISPATCH_ROS_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, {
      const int G = BLK / LPC;
      const unsigned need = (unsigned)((n + G - 1) / G);
      const unsigned cap = (unsigned)emp_resident<LPC, AR, BLK, 3>();
      hipLaunchKernelGGL((k_emp_adaptive2<LPC, AR, BLK>), dim3(need < cap ? need : cap), dim3(BLK), 0, st, d_dev,
                         list, n, d_params, d_ctl, next, pending, work, errflag);
    })));
    return true;
  }
  if (lpl != 1) return false;
  if (ros_selected(p)) {
    SC_DISPATCH_ROS_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, {
      const int G = BLK / LPC;
      const unsigned need = (unsigned)((n + G - 1) / G);
      const unsigned cap = (unsigned)emp_resident<LPC, AR, BLK, 2>();
      hipLaunchKernelGGL((k_ros_adaptive<LPC, AR, BLK>), dim3(need < cap ? need : cap), dim3(BLK), 0, st, d_dev,
                         list, n, d_params, d_ctl, next, pending, work, errflag);
    })));
    return true;
  }
  SC_DISPATCH_PW(p, SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, SC_DISPATCH_BLK(blk, {
    const int G = BLK / LPC;
    const unsigned need = (unsigned)((n + G - 1) / G);
    const unsigned cap = (unsigned)emp_resident<LPC, AR, BLK, PW>();
    hipLaunchKernelGGL((k_emp_adaptive<LPC, AR, BLK, PW>), dim3(need < cap ? need : cap), dim3(BLK), 0, st, d_dev,
                       list, n, d_params, d_ctl, next, pending, work, errflag);
  }))));
  return true;
}

__global__ void k_emp_begin(const int *list, int n, int r0, int *wrec, double *wrem, long long *watt)
{
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = list[i];
    wrec[c] = r0 - 1;
    wrem[c] = 0.0;
    watt[c] = 0;
  }
}

// zc from sequential sums of dz (init_grid :161-168), exp(100 k_l zc),
// exp(200 k_l zc), and the depth to the last layer's top (the cumdepth left by
// the light loop of get_rhs :593-598); one thread per column, in the
// oracle's operation order
__global__ void k_zw_geometry(Dev d, const int *list, int n, double k_l, double *e1, double *e2, double *cum)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = list[i];
  const int o = d.off[c], K = d.off[c + 1] - o;
  double zi = 0.0, cd = 0.0;
  for (int k = 0; k < K; ++k) {
    const double dz = d.dz[o + k];
    const double zc = zi + dz * 0.5;
    e1[o + k] = dexp((zc * 100.0) * k_l);
    e2[o + k] = dexp((zc * 200.0) * k_l);
    zi = zi + dz;
    if (k < K - 1) cd = cd + dz;
  }
  cum[c] = cd;
}

void launch_zw_geometry(hipStream_t st, const Dev &d, const int *list, int n, double k_l, double *e1, double *e2,
                        double *cum)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_zw_geometry, dim3((n + 255) / 256), dim3(256), 0, st, d, list, n, k_l, e1, e2, cum);
}

__global__ void k_fill_int(int *p, int n, int v)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_emp_begin(hipStream_t st, const int *list, int n, int r0, int *wrec, double *wrem, long long *watt)
{
  if (n <= 0) return;
  const int blocks = (n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024;
  hipLaunchKernelGGL(k_emp_begin, dim3(blocks), dim3(256), 0, st, list, n, r0, wrec, wrem, watt);
}

// ---------------------------------------------------------------------------
// warm start from log10 profiles on a geometric node grid
// ---------------------------------------------------------------------------

// ratio r of an n-layer geometric grid, dz1 (r^n - 1)/(r - 1) = total, by
// Newton's method on g(r) = dz1 (r^n - 1) - total (r - 1), which is convex
// for r > 0 with the roots 1 and the ratio.  A growing grid (n dz1 < total)
// has the larger root: from r0 = (total/dz1)^(1/(n-1)), where g(r0) =
// total - dz1 > 0, the iterates decrease monotonically onto it.  A
// shrinking grid has the smaller root: from r = 0 they increase onto it.
// The iteration stops when an iterate no longer moves in its direction
// (at most a few ulp from the root; the host's bisection lands as close).
__device__ double geometric_ratio_dev(int n, double dz1, double total)
{
  const double fn = (double)n;
  if (n <= 1 || fabs(fn * dz1 - total) <= 1e-15 * total) return 1.0;
  const bool grow = fn * dz1 < total;
  double r = grow ? pow(total / dz1, 1.0 / (fn - 1.0)) : 0.0;
  for (int it = 0; it < 100; ++it) {
    const double rm = pow(r, fn - 1.0);  // r^(n-1)
    const double g = dz1 * (rm * r - 1.0) - total * (r - 1.0);
    const double dg = (dz1 * fn) * rm - total;
    const double rn = r - g / dg;
    if (!(grow ? rn < r : rn > r)) break;
    r = rn;
  }
  return r;
}

// One column per group of LPC lanes, lane l = layer l.  The group builds
// the node centres in LDS (lanes stride over the nodes), then each layer
// interpolates every variable's profile at its own centre.
template <int LPC>
__global__ __launch_bounds__(BLOCK) void k_warm_profiles(Dev d, const int *list, int nlist, WarmProfiles w)
{
  constexpr int G = BLOCK / LPC;
  __shared__ double sdz[G][kWarmMaxNodes];
  __shared__ double szc[G][kWarmMaxNodes];
  const int g = threadIdx.x / LPC, l = threadIdx.x % LPC;
  const int slot = blockIdx.x * G + g;
  const bool live = slot < nlist;
  const int c = live ? list[slot] : 0;
  const int o = live ? d.off[c] : 0, K = live ? d.off[c + 1] - o : 0;
  if (live) {
    double depth = 0.0;
    if (w.depth)
      depth = w.depth[c];
    else
      for (int k = 0; k < K; ++k) depth = depth + d.dz[o + k];
    const double r = geometric_ratio_dev(w.nz, w.dz1, depth);
    for (int j = l; j < w.nz; j += LPC) sdz[g][j] = w.dz1 * pow(r, (double)j);
  }
  __syncthreads();
  if (live)
    for (int j = l; j < w.nz; j += LPC) {
      double zi = 0.0;
      for (int q = 0; q < j; ++q) zi = zi + sdz[g][q];
      szc[g][j] = zi + 0.5 * sdz[g][j];
    }
  __syncthreads();
  if (!live || l >= K) return;
  double zi = 0.0;
  for (int q = 0; q < l; ++q) zi = zi + d.dz[o + q];
  const double zk = zi + 0.5 * d.dz[o + l];
  int j = -1;
  for (int q = 0; q < w.nz; ++q) j += zk >= szc[g][q] ? 1 : 0;
  j = j < 0 ? 0 : (j > w.nz - 2 ? w.nz - 2 : j);
  const double z0 = szc[g][j], z1 = szc[g][j + 1];
  double wt = (zk - z0) / (z1 - z0);
  wt = wt < 0.0 ? 0.0 : (wt > 1.0 ? 1.0 : wt);
  const float *row = w.prof + (long long)c * w.ld;
  const long long cell = (long long)o + l;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i0 = n * w.nz + j;
    const double f0 = (double)row[i0] * w.scale[i0] + w.offset[i0];
    const double f1 = (double)row[i0 + 1] * w.scale[i0 + 1] + w.offset[i0 + 1];
    const double x = exp10(f0 + wt * (f1 - f0)) - w.eps[n];
    d.conc[n * d.ncell + cell] = x < 0.0 ? 0.0 : x;  // NaN stays NaN
  }
}

void launch_warm_profiles(int lpc, hipStream_t st, const Dev &d, const int *list, int n, const WarmProfiles &w)
{
  SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_warm_profiles<LPC>), grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n,
                                          w));
}

void launch_fill_int(hipStream_t st, int *p, int n, int v)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_int, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
}

__global__ void k_fill_dbl(double *p, long long n, double v)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_dbl(hipStream_t st, double *p, long long n, double v)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_dbl, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

// Fortran arrays f[(n K + k) ncol + c] against packed ones x[(n ncol + c) K + k]
// of a uniform grid, nvar planes: a transposition of ncol x K per plane.  64
// columns per block go through LDS, so that both sides are read and written in
// whole lines: rows of 64 columns of f, and one run of 64 K values of x (one
// thread per element, in Fortran order, wrote or read x with a stride of K:
// 32 us for 11 planes of 8000 columns of 30 layers, this 14 us; 90000 columns
// take 121 us, 3.9 TB/s).
constexpr int kLayoutCols = 64;
__global__ __launch_bounds__(256) void k_layout(const double *__restrict__ src, double *__restrict__ dst, int ncol,
                                                int K, int to_packed)
{
  __shared__ double tile[SEDCOL_KMAX][kLayoutCols + 1];
  const int c0 = blockIdx.x * kLayoutCols;
  const int nc = ncol - c0 < kLayoutCols ? ncol - c0 : kLayoutCols;
  const long long plane = (long long)ncol * K;
  const long long f0 = (long long)blockIdx.y * plane + c0;               // f of (k = 0, c0)
  const long long x0 = (long long)blockIdx.y * plane + (long long)c0 * K;  // x of (c0, k = 0)
  const int cc = threadIdx.x % kLayoutCols, kq = threadIdx.x / kLayoutCols;
  if (to_packed) {
    if (cc < nc)
      for (int k = kq; k < K; k += 256 / kLayoutCols) tile[k][cc] = src[f0 + (long long)k * ncol + cc];
    __syncthreads();
    for (int i = threadIdx.x; i < nc * K; i += 256) {
      const int c = i / K;
      dst[x0 + i] = tile[i - c * K][c];
    }
  } else {
    for (int i = threadIdx.x; i < nc * K; i += 256) {
      const int c = i / K;
      tile[i - c * K][c] = src[x0 + i];
    }
    __syncthreads();
    if (cc < nc)
      for (int k = kq; k < K; k += 256 / kLayoutCols) dst[f0 + (long long)k * ncol + cc] = tile[k][cc];
  }
}

void launch_layout(hipStream_t st, const double *src, double *dst, int ncol, int K, int nvar, bool to_packed)
{
  if (ncol <= 0 || K <= 0 || nvar <= 0) return;
  hipLaunchKernelGGL(k_layout, dim3((unsigned)((ncol + kLayoutCols - 1) / kLayoutCols), (unsigned)nvar), dim3(256), 0,
                     st, src, dst, ncol, K, to_packed ? 1 : 0);
}

// n doubles, and up to three small copies on the way: from, or to, pinned host
// memory that the device reads and writes in place
__global__ void k_stage(const double *__restrict__ src, double *__restrict__ dst, long long n, const double *s1,
                        double *d1, int n1, const int *s2, int *d2, int n2, int *zero)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
  if (i < n1) d1[i] = s1[i];
  if (i < n2) d2[i] = s2[i];
  if (zero && i == 0) *zero = 0;
}

void launch_stage(hipStream_t st, const double *src, double *dst, long long n, const double *s1, double *d1, int n1,
                  const int *s2, int *d2, int n2, int *zero)
{
  long long m = n > n1 ? n : n1;
  m = m > n2 ? m : n2;
  if (m < 1) m = 1;
  hipLaunchKernelGGL(k_stage, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, src, dst, n, s1, d1, n1, s2, d2,
                     n2, zero);
}

void launch_ae_rhs(int lpc, hipStream_t st, const Dev &d, const int *list, int n, const sedcol_params &p, int rec,
                   double dt_red, double *r_out, double *s_out, int *viol)
{
  SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_ae_rhs<LPC, AR>), grid_for<LPC>(n), dim3(BLOCK), 0,
                                                               st, d, list, n, p, rec, dt_red, r_out, s_out, viol)));
}

void launch_ae_check(int lpc, hipStream_t st, const Dev &d, const int *list, int n, double dt_red, double rcm,
                     const double *r_in, int *viol)
{
  SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_ae_check<LPC>), grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n,
                                          dt_red, rcm, r_in, viol));
}

void launch_ae_commit(int lpc, hipStream_t st, const Dev &d, const int *list, int n, double dt_red, double dt_min,
                      bool clamp, const double *r_in, const double *s_in, const int *viol, int *clear, int *errflag)
{
  SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_ae_commit<LPC>), grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n,
                                          dt_red, dt_min, clamp ? 1 : 0, r_in, s_in, viol, clear, errflag));
}

void launch_ae_fused(int lpc, hipStream_t st, const Dev *d_dev, const int *list, int n, const sedcol_params &p,
                     const sedcol_params *d_params, int rec, double dt, int nsteps, int *errflag, double *min_dt)
{
  // the smallest block that holds the columns: one wave, one wave per SIMD
  // (all registers), two
#define SC_AE_FUSED(BLK)                                                                                           \
  SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_ae_fused<LPC, AR, BLK>), dim3(1), dim3(BLK), 0, st, \
                                                                d_dev, list, n, d_params, rec, dt, nsteps, errflag, \
                                                                min_dt)))
  if (n * lpc <= 64) {
    SC_AE_FUSED(64);
  } else if (n * lpc <= 256) {
    SC_AE_FUSED(256);
  } else {
    SC_AE_FUSED(kAeFusedBlock);
  }
#undef SC_AE_FUSED
}

void launch_budget(int lpc, hipStream_t st, const Dev &d, const int *list, int n, double *budget)
{
  SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_budget<LPC>), grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n,
                                          budget));
}

void launch_inventory(int lpc, hipStream_t st, const Dev &d, const int *list, int n, double *inv)
{
  SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_inventory<LPC>), grid_for<LPC>(n), dim3(BLOCK), 0, st, d, list, n,
                                          inv));
}

void launch_residual(int lpc, hipStream_t st, const Dev &d, const int *list, int n, const sedcol_params &p, int rec,
                     const double *cfloor, double *resid, double *flux)
{
  SC_DISPATCH_ARITH(p, SC_DISPATCH_LPC(lpc, hipLaunchKernelGGL((k_residual<LPC, AR>), grid_for<LPC>(n), dim3(BLOCK),
                                                               0, st, d, list, n, p, rec, cfloor, resid, flux)));
}

}  // namespace sc
