// wg_kernels.hip -- HIP kernels for gfx950: the daily vertical water balance and
// the lateral routing of WaterGAP 2 (parity option profile).
//
// Calls of three days and more run wg_days_kernel (wg_days_kernel.h), one launch for
// many days.  Shorter ones run two kernels per simulated day, with the same per-cell
// functions (wg_cell_day.h, wg_route_step.h):
//   wg_cell_kernel   one lane per (member, cell).  It finishes the previous day
//                    (reduction factors, river width, surface-water and land area
//                    fractions: routing.cpp:2478-2488, 2792-2802, 3071-3078,
//                    3286-3295, 3546-3586, 5034-5188, 5343-5352), runs calcNewDay
//                    (daily.cpp:94-1279, lai.cpp:152-306) and the part of the
//                    routing loop that reads no upstream water (routing.cpp:1877-2617),
//                    and for cells without upstream cells the whole rest of the
//                    routing loop as well.
//   wg_chain_kernel  one workgroup per (routing group, member).  It walks the Kahn
//                    levels of the group with workgroup barriers; each cell gathers
//                    the transported volume of its upstream cells in routing order
//                    (the order of the serial += at routing.cpp:3955-3958) and runs
//                    routing.cpp:2623-3958 (global lake, reservoir, global wetland,
//                    arid groundwater, river).
// Arithmetic follows the reference expression by expression (operand order and
// association), compiled with -ffp-contract=off, in FP64 with the reference's
// float/short inputs promoted exactly where the reference promotes them; exp and
// pow are the deterministic ones of wg_libm.h, shared with the CPU oracle.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wg_device.h"
// The exp/log/pow table lives in LDS, one copy per wavefront at the front of the
// workgroup's dynamic LDS (WG_EXP2_LDS_BYTES per wavefront): a lane-varying index
// into a global table costs a vector-memory round trip per lookup, two per pow.
extern __shared__ double wg_lds[];
#define WG_EXP2_LDS_BYTES 1024
#define WG_EXP2_TAB_LDS (wg_lds + 128 * (threadIdx.x >> 6))
#include "wg_libm.h"

namespace {
// Copies the table into the wavefront's LDS copy with one direct global-to-LDS load
// (16 bytes per lane, lane i to bytes 16i..16i+15).  The compiler waits for it
// before the first LDS read.
__device__ inline void load_exp2_table() {
  const int lane = threadIdx.x & 63;
  __builtin_amdgcn_global_load_lds((const void *)(wg_exp2_tab_d + 2 * lane),
                                   (__attribute__((address_space(3))) void *)(wg_lds + 128 * (threadIdx.x >> 6)), 16, 0,
                                   0);
}
}  // namespace

namespace {

#include "wg_route_step.h"

// ---- ensemble perturbation: Philox4x32-10 + Box-Muller normal deviates ----
__device__ inline void philox(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; r++) {
    const uint32_t hi0 = __umulhi(0xD2511F53u, c[0]), lo0 = 0xD2511F53u * c[0];
    const uint32_t hi1 = __umulhi(0xCD9E8D57u, c[2]), lo1 = 0xCD9E8D57u * c[2];
    const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = lo1;
    c[2] = n2;
    c[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// Two independent standard normal deviates for (cell, day) of one member: one
// Philox block gives u1, u2 = (c + 1/2) 2^-32 in (0, 1); Box-Muller
// R = sqrt(-2 ln u1), z = (R cos 2 pi u2, R sin 2 pi u2).  ln, sin and cos are the
// deterministic ones shared with the host, sqrt is correctly rounded, so the
// oracle draws the same bits.  |z| < 6.7 (u1 >= 2^-33).
__device__ inline void normal_pair(uint64_t seed, uint32_t cell, uint32_t day, double &z0, double &z1) {
  uint32_t c[4] = {cell, day, 0x424f584du, 0u};
  philox(c, uint32_t(seed), uint32_t(seed >> 32));
  const double u1 = (double(c[0]) + 0.5) * 2.3283064365386963e-10;
  const double u2 = (double(c[1]) + 0.5) * 2.3283064365386963e-10;
  const double r = sqrt(-2.0 * wg_log(u1));
  double sn, cs;
  wg_sincos2pi(u2, &sn, &cs);
  z0 = r * cs;
  z1 = r * sn;
}

// Element i of a row that is the same for the whole wavefront: a scalar base and a
// 32-bit byte offset (rows hold fewer than 2^27 elements of up to 16 bytes).  The
// empty asm keeps the offset a 32-bit value of the block that uses it; otherwise the
// compiler forms every row's 64-bit address ahead of the day loop and spills them.
template <class T>
__device__ __forceinline__ T &at(T *row, uint32_t i) {
  uint32_t o = i * uint32_t(sizeof(T));
  asm volatile("" : "+v"(o));
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(const_cast<std::remove_const_t<T> *>(row)) + o);
}

// Device accessors of the routing links and chain constants ([k][N] x 16 bytes).
__device__ inline WgChainLink load_link(const WgStatic &S, uint32_t p) {
  const WgI4 a = at(S.clink, p), b = at(S.clink + S.n, p);
  WgChainLink lk;
  lk.flags = a.x;
  lk.station = a.y;
  lk.nu = int16_t(a.z & 0xffff);
  lk.nu_level = int16_t(a.z >> 16);
  lk.level = a.w;
  const int32_t u[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    lk.up[2 * k] = int16_t(uint32_t(u[k]) & 0xffff);
    lk.up[2 * k + 1] = int16_t(uint32_t(u[k]) >> 16);
  }
  return lk;
}

__device__ inline WgChainStatic load_cstat(const WgStatic &S, uint32_t p) {
  const int64_t n = S.n;
  const WgD2 a = at(S.cstat, p), b = at(S.cstat + n, p), c = at(S.cstat + 2 * n, p);
  return WgChainStatic{a.x, a.y, b.x, b.y, c.x, c.y};
}

// Writes what chain_step changed; o: the offset of the member's rows.
__device__ inline void store_chain(const WgState &X, int64_t o, uint32_t p, int flags, const ChainOut &r) {
  if (flags & CFL_LAKE) at(X.glo_lake + o, p) = r.glo_lake;
  if (flags & CFL_RES) {
    at(X.res + o, p) = r.res;
    at(X.k_release + o, p) = r.k_release;
  }
  if (flags & CFL_GWET) at(X.glo_wetl + o, p) = r.glo_wetl;
  if (flags & CFL_ARID) at(X.gw + o, p) = r.gw;
  if ((flags & CFL_ARID) && X.pot_lgw) at(X.pot_lgw + o, p) = r.lgw;
  at(X.river + o, p) = r.river;
  at(X.tv + o, p) = r.tv;
  if (X.use_rem) at(X.use_rem + o, p) = r.rem;
}

#include "wg_cell_day.h"

}  // namespace

namespace {

// Loads of a cell's statics and state, grouped by the part of the day that reads
// them.  A kernel issues a part's loads before the first store of that part, so
// that they are in flight together (after a store the compiler must keep later
// loads behind it).  Every array covers all cells, so the loads of fields a cell
// does not use are in bounds.
__device__ __forceinline__ void load_stat_a(const WgStatic &S, const WgTables &T, uint32_t p, DayStatA &a) {
  const int l = at(S.land_cover, p) - 1;
  const float lmax_f = at(S.lai_max, p);
  a.m_prec = at(S.m_prec, p);
  a.alpha = at(S.alpha, p);
  a.pet_mxdy = at(S.pet_mxdy, p);
  a.m_netrad = at(S.m_netrad, p);
  a.mcwh = at(S.mcwh, p);
  a.t_snowfz = at(S.t_snowfz, p);
  a.t_snowmt = at(S.t_snowmt, p);
  a.t_gradnt = at(S.t_gradnt, p);
  a.melt_factor = at(S.degday, p) * T.ddf[l];
  a.albedo = T.albedo[l];
  a.albedo_snow = T.albedo_snow[l];
  a.emis = T.emissivity[l] * 0.000000004903;
  a.lmin = T.lai_a[l] + T.lai_b[l] * lmax_f;
  a.lmax = lmax_f;
  a.initial_days = T.initial_days[l];
  a.lct = l + 1;
  a.elev0 = at(S.elev0, p);
  a.arid = at(S.aindex, p) == 1;
}

__device__ __forceinline__ void load_stat_b(const WgStatic &S, const WgState &X, int64_t o, uint32_t p, DayStatB &b) {
  b.built_up = at(S.built_up, p);
  b.smax = at(X.smax + o, p);
  b.gw_factor = at(S.gw_factor, p);
  b.gamma = at(X.gamma + o, p);
  b.cfa = at(X.cfa + o, p);
  b.pet_mxdy = at(S.pet_mxdy, p);
  b.t_snowfz = at(S.t_snowfz, p);
  b.pcritgwa = at(S.pcritgwa, p);
  const int16_t rgmax = at(S.rgmax, p);
  b.rgmax = rgmax / 100.;
  b.arid = at(S.aindex, p) == 1;
  b.ldd = at(S.ldd, p);
  b.recharge_cut = (b.arid && (at(S.texture, p) < 21)) && (b.ldd >= 0);
  b.area = at(S.cell_area, p);
  b.area_m = b.area / 1000000.;
  b.cf100 = at(S.contfreq, p) / 100.;
  double f = at(S.fswb_init, p) * 20.;
  if (f > 1.) f = 1.;
  b.fswb_catchment = f;
  b.e_gw = at(S.e_gw, p);
  b.inv_kgw = at(S.inv_kgw, p);
  b.ome_gw = at(S.ome_gw, p);
  b.e_sw = at(S.e_sw, p);
  b.k_sw = at(S.k_sw, p);
  b.red_exp = at(S.evarexp, p) * kEvapoRedExp;
  const double lake_depth = at(S.lake_depth, p), wetl_depth = at(S.wetl_depth, p);
  b.loc_lake = at(S.loc_lake, p);
  b.ll100 = b.loc_lake / 100.;
  b.ll_max = b.ll100 * b.area * lake_depth;
  b.loc_wetland = at(S.loc_wetland, p);
  b.lw100 = b.loc_wetland / 100.;
  b.lw_max = b.lw100 * b.area * wetl_depth;
  b.glo_wetland = at(S.glo_wetland, p);
  b.gw100 = b.glo_wetland / 100.;
  b.gw_max = b.gw100 * b.area * wetl_depth;
  b.river_length = at(S.river_length, p);
  b.bottom = at(S.bottom_width, p);
  b.vel_b4 = -b.bottom / 4.0;
  b.vel_b16 = b.bottom * b.bottom / 16.0;
  b.vel_c1 = at(S.vel_c1, p);
  b.vel_c2 = at(S.vel_c2, p);
}

__device__ __forceinline__ void load_stat_lake(const WgStatic &S, uint32_t p, DayStatLake &k) {
  k.lake_area = at(S.lake_area, p);
  k.lake_depth = at(S.lake_depth, p);
  k.reservoir_area = at(S.reservoir_area, p);
  k.stor_cap = at(S.stor_cap, p);
  k.mean_outflow = at(S.mean_outflow, p);
  k.prov_rel = at(S.res_prov_rel, p);
}

__device__ __forceinline__ void load_stat_end(const WgStatic &S, uint32_t p, DayStatEnd &e) {
  e.red_exp = at(S.evarexp, p) * kEvapoRedExp;
  e.area = at(S.cell_area, p);
  e.river_length = at(S.river_length, p);
  e.rw_c0 = at(S.rw_c0, p);
  e.rw_c1 = at(S.rw_c1, p);
  e.rw_c2 = at(S.rw_c2, p);
  e.rw_c3 = at(S.rw_c3, p);
  e.river_stor_max = at(S.river_stor_max, p);
  e.f_glo_lake = at(S.f_glo_lake, p);
  e.max_raf = at(S.contfreq, p) / 100. - e.f_glo_lake;
  e.loc_lake = at(S.loc_lake, p);
  e.loc_wetland = at(S.loc_wetland, p);
  e.glo_wetland = at(S.glo_wetland, p);
  e.gw_max = e.glo_wetland / 100. * e.area * at(S.wetl_depth, p);
  e.lake_area = at(S.lake_area, p);
  e.lake_max = e.lake_area * at(S.lake_depth, p);
  e.reservoir_area = at(S.reservoir_area, p);
  e.stor_cap = at(S.stor_cap, p);
  e.contcell = at(S.contcell, p) != 0;
}

__device__ __forceinline__ ElevRange load_elev_range(const WgStatic &S, uint32_t p) {
  const int32_t r = at(S.elev_range, p), e = at(S.elev_pairs, p);
  return ElevRange{int16_t(r & 0xffff), int16_t(r >> 16), int16_t(e & 0xffff)};
}

// State read by PET, LAI, canopy and snow.
__device__ __forceinline__ void load_state_a(const WgState &X, int64_t o, uint32_t p, CellState &s) {
  s.canopy = at(X.canopy + o, p);
  s.lai_days = at(X.lai_days + o, p);
  s.lai_precsum = at(X.lai_precsum + o, p);
  s.lai_status = at(X.lai_status + o, p);
  s.snow = at(X.snow + o, p);
  s.snow_any = at(X.snow_any + o, p) != 0;
  s.transfer = at(X.transfer + o, p);
}

// State read by soil and local routing.
__device__ __forceinline__ void load_state_b(const WgState &X, int64_t o, uint32_t p, CellState &s) {
  s.soil = at(X.soil + o, p);
  s.gw = at(X.gw + o, p);
  s.loc_lake = at(X.loc_lake + o, p);
  s.loc_wetl = at(X.loc_wetl + o, p);
  s.glo_lake = at(X.glo_lake + o, p);
  s.glo_wetl = at(X.glo_wetl + o, p);
  s.res = at(X.res + o, p);
  s.river = at(X.river + o, p);
  s.k_release = at(X.k_release + o, p);
}

// State read by the day's end (with loc_lake for the water use).
__device__ __forceinline__ void load_state_end(const WgState &X, int64_t o, uint32_t p, CellState &s) {
  s.glo_lake = at(X.glo_lake + o, p);
  s.glo_wetl = at(X.glo_wetl + o, p);
  s.res = at(X.res + o, p);
  s.river = at(X.river + o, p);
  s.red_ll = at(X.red_ll + o, p);
  s.red_lw = at(X.red_lw + o, p);
  s.red_gl = 0.;
  s.red_gw = at(X.red_gw + o, p);
  s.red_res = 0.;
  s.red_river = at(X.red_river + o, p);
  s.river_frac_next = at(X.river_frac_next + o, p);
  s.river_frac_change = at(X.river_frac_change + o, p);
  s.fswb_next = at(X.fswb_next + o, p);
  s.laf = at(X.laf + o, p);
}

// Writes what the day's end changed.
__device__ __forceinline__ void store_state_end(const WgState &X, int64_t o, uint32_t p, const DayStatEnd &e,
                                                const CellState &s) {
  if (e.lake_area > 0.) at(X.red_gl + o, p) = s.red_gl;
  if (e.reservoir_area > 0.) at(X.red_res + o, p) = s.red_res;
  at(X.laf_prev + o, p) = s.laf_prev;
  at(X.laf + o, p) = s.laf;
  at(X.fswb_next + o, p) = s.fswb_next;
  at(X.red_ll + o, p) = s.red_ll;
  at(X.red_lw + o, p) = s.red_lw;
  at(X.red_gw + o, p) = s.red_gw;
  at(X.red_river + o, p) = s.red_river;
  at(X.river_frac_next + o, p) = s.river_frac_next;
  at(X.river_frac_change + o, p) = s.river_frac_change;
}

// The day's perturbed temperature and precipitation of one (member, cell).
__device__ __forceinline__ void perturb_forcing(const WgStatic &S, const WgState &X, int m, uint32_t p, int64_t fday,
                                                float &tf, float &pf) {
  const uint64_t seed = X.member_seed[m];
  const uint32_t ref = uint32_t(at(S.ref_index, p));
  double zp, zt;
  normal_pair(seed, ref, uint32_t(fday), zp, zt);
  pf = float(double(pf) * wg_exp(X.prec_sigma * zp));
  tf = float(double(tf) + X.temp_sigma * zt);
}

// Water use of the day: the desired surface-water use (routing.cpp:2193-2290) and
// the net abstraction from groundwater (routing.cpp:7440-7441, adapted by
// updateNetAbstractionGW in every groundwater branch when the last day left a
// remaining use; the adaptation reads only the last day's state, so it is done
// here for (semi-)arid cells too, whose groundwater step the chain runs).
// Returns the offset of the day's rows in the tables.
__device__ __forceinline__ int64_t day_use(const WgStatic &S, const WgState &X, int64_t o, uint32_t p, int64_t fday,
                                           int month, double &desired, double &nag) {
  const int64_t t = (int64_t((fday - S.use_day0) / 365) * 12 + month) * S.n;
  const int64_t us = S.use_stride;
  double *U = X.use + o;
  nag = at(S.use_nug + t, p);
  if (at(U + WG_USE_DAILY_REMAINING * us, p) != 0.) nag = update_net_abstraction_gw(U, us, p, at(S.use_frgi, p), nag);
  desired = at(S.use_nus + t, p);
  if (S.use_delayed == 1) desired += at(U + WG_USE_TOTAL_UNSAT * us, p);
  return t;
}

// Adds the day's potential cell runoff of a continental cell to its running sum,
// G_potCellRunoff[n] += potCellRunoff (routing.cpp:1970, 2053, 2187, 3379): the
// local runoff terms, then the arid groundwater step's runoff where that step ran,
// then the open-water balance, in the reference's order of addition.
__device__ __forceinline__ void add_pot_runoff(const WgStatic &S, const WgState &X, int64_t o, uint32_t p) {
  const double base = at(X.pot_base + o, p);
  const double lake_balance = at(X.pot_ow + o, p) * at(X.cfa + o, p);  // (dailyPrec - dailyOpenWaterPET) * CFA
  const double ow = (lake_balance / 1000000.0) *
                    ((at(S.lake_area, p) + at(S.reservoir_area, p)) +
                     ((at(S.cell_area, p) / 100.0) * ((at(S.loc_lake, p) + at(S.loc_wetland, p)) + at(S.glo_wetland, p))));
  const double pot = (at(S.cflags, p) & CFL_ARID) ? (base + at(X.pot_lgw + o, p)) + ow : base + ow;
  at(X.pot_acc + o, p) += pot;
}

}  // namespace

struct WgClock {
  int64_t day0;   // forcing day (index into the loaded forcing) of launch offset 0
  int32_t doy0;   // julian day of launch offset 0
  int32_t started;
};

// One lane per (member, cell).  Grid: x over cell tiles, y over members.
// kSnowChunk: sub-cell pairs per chunk of the snow loop (5 or 10).
// With chunks of 5 pairs the kernel is held to 168 registers, three wavefronts per
// SIMD, for many members, where it is bandwidth-bound; chunks of 10 leave the
// compiler free, for one member, where it is latency-bound.
// kUse: water use on (the handle's tables are set); the instantiation without it
// is the model without water use, with no use code at all.
template <int kSnowChunk, bool kUse>
__global__ __launch_bounds__(256, kSnowChunk == 5 ? 3 : 1) void wg_cell_kernel(WgStatic S, WgState X, WgTables T,
                                                      const float *__restrict__ forcing, int64_t n_forcing_days,
                                                      const WgClock *__restrict__ clock, int k,
                                                      int do_post, int do_vertical, int write_diag,
                                                      int daily_slot) {
  load_exp2_table();
  const int t0 = S.tile_start[blockIdx.x];
  if (t0 < 0) return;
  const uint32_t p = uint32_t(t0) + threadIdx.x;
  if (int(p) >= S.tile_end[blockIdx.x]) return;
  const int m = blockIdx.y;
  const int n = S.n;
  const int64_t o = int64_t(m) * n;

  DayStatA sa;
  CellState s;
  ElevRange er{0, 0, 0};
  if (do_vertical) {
    er = load_elev_range(S, p);
    load_stat_a(S, T, p, sa);
    load_state_a(X, o, p, s);
  }
  if (do_post) {
    DayStatEnd e;
    load_stat_end(S, p, e);
    load_state_end(X, o, p, s);
    if (kUse && e.contcell) {
      // the finished day is day k - 1 of the block (the closing pass runs with k = days)
      const int64_t fin = clock->day0 + k - 1;
      const int fin_doy = int((clock->doy0 - 1 + k - 1) % 365) + 1;
      const int fin_ym = int((fin - S.use_day0) / 365) * 12 + day_info(fin_doy).month;
      s.loc_lake = at(X.loc_lake + o, p);
      day_end_use(S, X.use + o, p, s, at(X.use_rem + o, p), e.loc_lake,
                  e.loc_lake / 100. * e.area * at(S.lake_depth, p), e.red_exp, fin_ym, fin_doy == 365);
      at(X.loc_lake + o, p) = s.loc_lake;
      at(X.use_rem + o, p) = 0.;
    }
    day_end(e, s);
    store_state_end(X, o, p, e, s);
  } else if (do_vertical) {
    s.laf = at(X.laf + o, p);
    s.laf_prev = at(X.laf_prev + o, p);
    s.red_ll = at(X.red_ll + o, p);
    s.red_lw = at(X.red_lw + o, p);
    s.red_gw = at(X.red_gw + o, p);
    s.red_gl = at(X.red_gl + o, p);
    s.red_res = at(X.red_res + o, p);
    s.river_frac_next = at(X.river_frac_next + o, p);
  }
  // calcNewDay and routing run for continental cells only (integrateWGHM.cpp:770,
  // routing.cpp:1876); other cells keep a zero transported volume.
  if (!do_vertical) return;
  if (!at(S.contcell, p)) {
    const int st = at(S.station, p);
    if (st >= 0) X.st_daily[(int64_t(m) * WG_DAILY_SLOTS + daily_slot) * S.n_stations + st] = 0.;
    return;
  }

  const int64_t fday = clock->day0 + k;
  const int doy = int((clock->doy0 - 1 + k) % 365) + 1;
  const bool started = (clock->started != 0) || (k > 0) || (do_post != 0);
  if (fday < 0 || fday >= n_forcing_days) return;
  const float *f = forcing + fday * 4 * int64_t(n);
  float tf = at(f, p), pf = at(f + n, p);
  const float swf = at(f + 2 * int64_t(n), p), lwf = at(f + 3 * int64_t(n), p);
  if (X.perturb) perturb_forcing(S, X, m, p, fday, tf, pf);
  double use_desired = 0., use_nag = 0.;
  int64_t use_t = 0;
  if (kUse) use_t = day_use(S, X, o, p, fday, day_info(doy).month, use_desired, use_nag);

  const double laf_prev = started ? s.laf_prev : s.laf;  // daily.cpp:159-169
  DayFlux v;
  day_pet_canopy(sa, s, v, tf, pf, swf, lwf, laf_prev);
  at(X.lai_days + o, p) = s.lai_days;
  at(X.lai_status + o, p) = s.lai_status;
  at(X.lai_precsum + o, p) = s.lai_precsum;
  at(X.canopy + o, p) = s.canopy;
  if (s.laf <= 0.)
    day_snow_no_land(s, v, X.snow2 + o * WG_DEV_NPAIR, p, n);
  else
    day_snow<kSnowChunk, false>(sa, s, v, laf_prev, er, X.snow2 + o * WG_DEV_NPAIR, S.elev_pairs, p, n);
  at(X.snow_any + o, p) = s.snow_any ? 1 : 0;
  DayStatB sb;
  DayStatLake lake;
  load_stat_b(S, X, o, p, sb);
  load_stat_lake(S, p, lake);
  load_state_b(X, o, p, s);
  const WgChainLink lk = load_link(S, p);
  const WgChainStatic cs = load_cstat(S, p);
  if (kUse) lake.prov_rel = at(S.use_provrel + use_t, p);
  at(X.snow + o, p) = s.snow;
  day_soil(sb, s, v, laf_prev);
  at(X.soil + o, p) = s.soil;
  at(X.transfer + o, p) = s.transfer;
  if (write_diag) {
    at(X.d_surf + o, p) = v.surf_runoff;
    at(X.d_recharge + o, p) = v.recharge;
    at(X.d_ow_pet + o, p) = v.ow_pet;
    at(X.d_aet + o, p) = v.aet;
    at(X.d_prec + o, p) = v.prec;
  }
  ChainRec c;
  double *w = c.v;
  c.inv_ksw = cs.inv_ksw;
  c.ome_sw = cs.ome_sw;
  c.inv_kgw = cs.inv_kgw;
  c.ome_gw = cs.ome_gw;
  c.area = cs.area;
  c.cf100 = cs.cf100;
  c.flags = lk.flags;
  PotTerms pot;
  day_local_routing<kUse>(sb, lake, s, v, use_desired, use_nag, c, pot);
  if (!(sb.arid && (sb.ldd >= 0))) at(X.gw + o, p) = s.gw;
  if (X.pot_base) {
    at(X.pot_base + o, p) = pot.base;  // wg_pot_runoff_kernel completes the terms
    at(X.pot_ow + o, p) = pot.ow;
  }
  if (sb.loc_lake > 0.) {
    at(X.loc_lake + o, p) = s.loc_lake;
    at(X.red_ll + o, p) = s.red_ll;
  }
  if (sb.loc_wetland > 0.) {
    at(X.loc_wetl + o, p) = s.loc_wetl;
    at(X.red_lw + o, p) = s.red_lw;
  }
  if (lk.nu == 0) {
    // no upstream cell: G_riverInflow[n] is still 0 when the cell is routed
    const ChainOut r = chain_step<kUse>(c, 0.0, day_info(doy));
    store_chain(X, o, p, c.flags, r);
    if (lk.station >= 0)
      X.st_daily[(int64_t(m) * WG_DAILY_SLOTS + daily_slot) * S.n_stations + lk.station] = (sb.ldd >= 0) ? r.tv : 0.;
  } else {
    // the pairs holding the prefix for every routed cell (the last of them also
    // holds the first suffix field), the rest for cells with a lake or reservoir
    constexpr int kPrefixPairs = (CF_PREFIX + 1) / 2;
#pragma unroll
    for (int k = 0; k < kPrefixPairs; k++) at(X.crec + o * (WG_DEV_NREC / 2) + int64_t(k) * n, p) = WgD2{w[2 * k], w[2 * k + 1]};
    if (lk.flags & (CFL_LAKE | CFL_RES)) {
#pragma unroll
      for (int k = kPrefixPairs; k < CF_USE / 2; k++) at(X.crec + o * (WG_DEV_NREC / 2) + int64_t(k) * n, p) = WgD2{w[2 * k], w[2 * k + 1]};
    }
    if (kUse) at(X.crec + o * (WG_DEV_NREC / 2) + int64_t(CF_USE / 2) * n, p) = WgD2{w[CF_USE], w[CF_A_NUG]};
  }
}

#include "wg_days_kernel.h"

// Workgroup barrier that orders LDS only.  The level walk exchanges data between
// threads through LDS alone (its global stores are read by later kernels), and a
// full __syncthreads() would also wait for the next level's prefetch loads
// (vmcnt counts loads and stores alike on this architecture).
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Inputs of one chain cell, loaded a level (or two) before it is routed: the
// whole routing record, the outflow constants and the links.  The record suffix
// holds data only for cells with a global lake or reservoir; it is loaded for
// every cell (so that no load depends on the flags) and zeroed for the others.
struct ChainSlot {
  double a[CF_COUNT];
  double inv_ksw, ome_sw, inv_kgw, ome_gw, area, cf100;
  int flags, nu, station, level, nu_level;
  int up[4];  // group-local upstream indices, two int16 per word
};

__device__ inline void prefetch_slot(const WgStatic &S, const WgState &X, int64_t base, int p, ChainSlot &q) {
  const int64_t n = S.n;
  const WgChainStatic cs = load_cstat(S, p);
  const WgD2 *src = X.crec + base * (WG_DEV_NREC / 2) + p;  // rec_at(X, n, m, p) for base = m * n
#pragma unroll
  for (int k = 0; k < CF_COUNT / 2; k++) {
    const WgD2 v = src[k * n];
    q.a[2 * k] = v.x;
    q.a[2 * k + 1] = v.y;
  }
  q.inv_ksw = cs.inv_ksw;
  q.ome_sw = cs.ome_sw;
  q.inv_kgw = cs.inv_kgw;
  q.ome_gw = cs.ome_gw;
  q.area = cs.area;
  q.cf100 = cs.cf100;
  const WgI4 a = S.clink[p], b = S.clink[n + p];
  q.flags = a.x;
  q.station = a.y;
  q.nu = a.z & 0xffff;
  q.nu_level = a.z >> 16;
  q.level = a.w;
  q.up[0] = b.x;
  q.up[1] = b.y;
  q.up[2] = b.z;
  q.up[3] = b.w;
}

typedef unsigned int WgU32x4 __attribute__((ext_vector_type(4)));

// Wave-walk variant of prefetch_slot: the record suffix is fetched only for cells
// with a global lake or reservoir (about 1.5 % of routed cells).  The cell's chain
// flags `fl` come from LDS, so no global load waits for another.  The other lanes
// issue the same suffix loads through raw buffers at an offset past the row's end,
// which the hardware answers with zeros without a memory access: every lane issues
// the same loads whatever its flags, so the count of outstanding loads, which the
// compiler's waits rely on, does not depend on them.
template <bool kUse>
__device__ inline void prefetch_slot_wave(const WgStatic &S, const WgState &X, int64_t base, int p, int fl,
                                          ChainSlot &q) {
  const int64_t n = S.n;
  const WgChainStatic cs = load_cstat(S, p);
  const WgD2 *src = X.crec + base * (WG_DEV_NREC / 2) + p;
  constexpr int kPrefixPairs = (CF_PREFIX + 1) / 2;
#pragma unroll
  for (int k = 0; k < kPrefixPairs; k++) {
    const WgD2 v = src[k * n];
    q.a[2 * k] = v.x;
    q.a[2 * k + 1] = v.y;
  }
  const bool suffix = (fl & (CFL_LAKE | CFL_RES)) != 0;
  const int off = suffix ? p * 16 : int(0x80000000u);
  WgD2 *row0 = X.crec + base * (WG_DEV_NREC / 2);
#pragma unroll
  for (int k = kPrefixPairs; k < CF_USE / 2; k++) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(row0 + k * n, (short)0, int(n * 16), 0x00020000);
    const WgU32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    q.a[2 * k] = __builtin_bit_cast(double, (unsigned long long)w.x | ((unsigned long long)w.y << 32));
    q.a[2 * k + 1] = __builtin_bit_cast(double, (unsigned long long)w.z | ((unsigned long long)w.w << 32));
  }
  // the water-use pair, for every cell when water use is on
  if (kUse) {
    const WgD2 u = src[int64_t(CF_USE / 2) * n];
    q.a[CF_USE] = u.x;
    q.a[CF_A_NUG] = u.y;
  } else {
    q.a[CF_USE] = 0.;
    q.a[CF_A_NUG] = 0.;
  }
  q.inv_ksw = cs.inv_ksw;
  q.ome_sw = cs.ome_sw;
  q.inv_kgw = cs.inv_kgw;
  q.ome_gw = cs.ome_gw;
  q.area = cs.area;
  q.cf100 = cs.cf100;
  const WgI4 a = S.clink[p], b = S.clink[n + p];
  q.flags = a.x;
  q.station = a.y;
  q.nu = a.z & 0xffff;
  q.nu_level = a.z >> 16;
  q.level = a.w;
  q.up[0] = b.x;
  q.up[1] = b.y;
  q.up[2] = b.z;
  q.up[3] = b.w;
}

// Wide-level variant: a batch of one level takes the record suffix when one of
// its cells has a global lake or reservoir (`suffix`, uniform over the wavefront,
// from the batch table), and issues no suffix loads otherwise.  Lake and reservoir
// cells come last in their level, so most batches load the prefix alone.  The
// workgroup's wavefronts share one CU's vector memory pipeline, which bounds the
// wide levels: every load instruction left out shortens them.
template <bool kUse>
__device__ inline void prefetch_slot_batch(const WgStatic &S, const WgState &X, int64_t base, int p, bool suffix,
                                           ChainSlot &q) {
  const int64_t n = S.n;
  const WgChainStatic cs = load_cstat(S, p);
  const WgD2 *src = X.crec + base * (WG_DEV_NREC / 2) + p;
  constexpr int kPrefixPairs = (CF_PREFIX + 1) / 2;
#pragma unroll
  for (int k = 0; k < kPrefixPairs; k++) {
    const WgD2 v = src[k * n];
    q.a[2 * k] = v.x;
    q.a[2 * k + 1] = v.y;
  }
  if (suffix) {
#pragma unroll
    for (int k = kPrefixPairs; k < CF_USE / 2; k++) {
      const WgD2 v = src[k * n];
      q.a[2 * k] = v.x;
      q.a[2 * k + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int k = 2 * kPrefixPairs; k < CF_USE; k++) q.a[k] = 0.;
  }
  if (kUse) {
    const WgD2 u = src[int64_t(CF_USE / 2) * n];
    q.a[CF_USE] = u.x;
    q.a[CF_A_NUG] = u.y;
  } else {
    q.a[CF_USE] = 0.;
    q.a[CF_A_NUG] = 0.;
  }
  q.inv_ksw = cs.inv_ksw;
  q.ome_sw = cs.ome_sw;
  q.inv_kgw = cs.inv_kgw;
  q.ome_gw = cs.ome_gw;
  q.area = cs.area;
  q.cf100 = cs.cf100;
  const WgI4 a = S.clink[p], b = S.clink[n + p];
  q.flags = a.x;
  q.station = a.y;
  q.nu = a.z & 0xffff;
  q.nu_level = a.z >> 16;
  q.level = a.w;
  q.up[0] = b.x;
  q.up[1] = b.y;
  q.up[2] = b.z;
  q.up[3] = b.w;
}

// The routing record of a slot (the suffix of a cell without a global lake or
// reservoir holds no data; chain_step does not read it for such cells).
__device__ inline void slot_record(const ChainSlot &q, ChainRec &c) {
#pragma unroll
  for (int f = 0; f < CF_COUNT; f++) c.v[f] = q.a[f];
  c.inv_ksw = q.inv_ksw;
  c.ome_sw = q.ome_sw;
  c.inv_kgw = q.inv_kgw;
  c.ome_gw = q.ome_gw;
  c.area = q.area;
  c.cf100 = q.cf100;
  c.flags = q.flags;
}

// Stores of the level walk.  Every lane issues the same stores on every level,
// whether or not it has a cell there and whatever storages the cell has: a store
// that must not land goes through a raw buffer over the destination row at an
// offset past the row's end, which the hardware drops.  A store behind a branch
// would leave different counts of outstanding memory operations on the two sides
// of the branch; the compiler's wait for the next level's inputs must then assume
// the smaller count, and waits for the loads just issued for the level after
// (loads and stores share one in-order counter on this architecture).
typedef unsigned int WgU32x2 __attribute__((ext_vector_type(2)));
// s_waitcnt immediate of the gfx9 family for vmcnt(0) (expcnt and lgkmcnt at their
// maxima, i.e. not waited on)
constexpr int kWaitVmcnt0 = 0x0F70;
constexpr uint32_t kDropOffset = 0x80000000u;  // past every row (rows hold < 2^28 doubles)

__device__ inline __amdgpu_buffer_rsrc_t row_buffer(double *row, int n) {
  // raw buffer (stride 0) of n doubles; the descriptor's last word is the one the
  // gfx9 family takes for untyped 32-bit dword access
  return __builtin_amdgcn_make_buffer_rsrc(row, (short)0, n * 8, 0x00020000);
}

__device__ inline void store_or_drop(double *row, int n, bool keep, int i, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(WgU32x2, v), row_buffer(row, n),
                                        int(keep ? uint32_t(i) * 8u : kDropOffset), 0, 0);
}

// One chain cell: ordered gather of the upstream transported volumes (the serial
// += of routing.cpp:3955-3958, in routing order), the upstream-dependent routing
// step, LDS and global stores, the station's daily discharge.  `act` is false for
// a lane without a cell on this level (its slot holds some other cell of the
// group, its results are not stored).
template <bool kUse>
__device__ __forceinline__ void chain_cell(const WgStatic &S, const WgState &X, double *s_tv, const ChainSlot &q,
                                           bool act, int64_t base, int p, int gs, int m, const DayInfo &d,
                                           int daily_slot) {
  const bool run = act && (q.flags & CFL_CONT);
  double up = 0.;
#pragma unroll
  for (int u = 0; u < 8; u++)
    if (u < q.nu) up += s_tv[(q.up[u >> 1] >> ((u & 1) * 16)) & 0xffff];
  ChainRec c;
  slot_record(q, c);
  const ChainOut o = chain_step<kUse>(c, up, d);
  const int n = S.n;
  store_or_drop(X.glo_lake + base, n, run && (q.flags & CFL_LAKE), p, o.glo_lake);
  store_or_drop(X.res + base, n, run && (q.flags & CFL_RES), p, o.res);
  store_or_drop(X.k_release + base, n, run && (q.flags & CFL_RES), p, o.k_release);
  store_or_drop(X.glo_wetl + base, n, run && (q.flags & CFL_GWET), p, o.glo_wetl);
  store_or_drop(X.gw + base, n, run && (q.flags & CFL_ARID), p, o.gw);
  if (X.pot_lgw) store_or_drop(X.pot_lgw + base, n, run && (q.flags & CFL_ARID), p, o.lgw);
  if (kUse) store_or_drop(X.use_rem + base, n, run, p, o.rem);
  store_or_drop(X.river + base, n, run, p, o.river);
  store_or_drop(X.tv + base, n, run, p, o.tv);
  if (run) s_tv[p - gs] = o.tv;
  const double qq = (run && (q.flags & CFL_LDD)) ? o.tv : 0.;
  store_or_drop(X.st_daily + (int64_t(m) * WG_DAILY_SLOTS + daily_slot) * S.n_stations, S.n_stations,
                act && q.station >= 0, q.station, qq);
}

// The first cell of level lf at this thread's position, or the group's first cell
// when there is none (or lf is past the group): the slot is loaded either way.
__device__ inline int slot_cell(const int32_t *__restrict__ lo, int lf, int l1, int gs) {
  const int lc = min(lf, l1 - 1);
  const int p = lo[lc] + int(threadIdx.x);
  return (lf < l1 && p < lo[lc + 1]) ? p : gs;
}

// One level of a group: the thread's first cell comes from `use` (loaded kAhead
// levels earlier); the first cell of level l + kAhead is loaded into `fill`
// before any computation, so its latency overlaps the levels in between.  The
// slots rotate by name, never copied, so no wait on the new loads is forced.
// Cells beyond the block size (levels wider than the block) load directly.
template <int kAhead, bool kUse>
__device__ __forceinline__ void chain_level(const WgStatic &S, const WgState &X, double *s_tv,
                                            const int32_t *__restrict__ lo, int l, int l1, int64_t base, int gs,
                                            int m, const DayInfo &d, int daily_slot, const ChainSlot &use,
                                            ChainSlot &fill) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int beg = lo[l], end = lo[l + 1];
  prefetch_slot(S, X, base, slot_cell(lo, l + kAhead, l1, gs), fill);
  const bool act = beg + tid < end;
  chain_cell<kUse>(S, X, s_tv, use, act, base, act ? beg + tid : gs, gs, m, d, daily_slot);
  for (int p = beg + tid + nt; p < end; p += nt) {
    ChainSlot q;
    prefetch_slot(S, X, base, p, q);
    chain_cell<kUse>(S, X, s_tv, q, true, base, p, gs, m, d, daily_slot);
  }
  lds_barrier();
}

// One workgroup per (routing group, member): levels 1..depth of the group.  The
// transported volumes of the group live in LDS (level 0 is copied in from the
// cell kernel's output); the static record holds group-local upstream indices.
// Each thread's first cell of a level is loaded kAhead levels early (1 or 2), so
// that the load latency overlaps the levels in between; the slots rotate by name.
template <int kAhead, bool kUse>
__global__ __launch_bounds__(256) void wg_chain_kernel(WgStatic S, WgState X, WgTables T,
                                                       const int32_t *__restrict__ group_level_off,
                                                       const int32_t *__restrict__ group_first_level,
                                                       const WgClock *__restrict__ clock, int k,
                                                       int daily_slot) {
  extern __shared__ double s_tv[];
  const int g = S.block_group[blockIdx.x];
  if (g < 0) return;
  const int m = blockIdx.y;
  const int n = S.n;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int doy = int((clock->doy0 - 1 + k) % 365) + 1;
  const DayInfo d = day_info(doy);
  const int32_t *lo = group_level_off;
  const int l0 = group_first_level[g], l1 = group_first_level[g + 1];
  const int gs = lo[l0], ge = lo[l1];
  if (l1 - l0 < 2 || ge <= gs) return;  // nothing routed in this kernel
  const int lvl0_end = lo[l0 + 1];
  const int64_t base = int64_t(m) * n;
  ChainSlot a, b, c;
  prefetch_slot(S, X, base, slot_cell(lo, l0 + 1, l1, gs), a);
  if (kAhead == 2) prefetch_slot(S, X, base, slot_cell(lo, l0 + 2, l1, gs), b);
  // level 0 was routed by the cell kernel; cells not routed today read as 0.
  // Eight loads in flight per thread before their LDS stores.
  for (int i0 = gs + tid; i0 < ge; i0 += 8 * nt) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int i = i0 + j * nt;
      v[j] = (i < lvl0_end) ? X.tv[base + i] : 0.;
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int i = i0 + j * nt;
      if (i < ge) s_tv[i - gs] = v[j];
    }
  }
  // the first slots' loads complete here on every path into the level loop, so
  // that the loop's waits count only what the loop itself issues
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  lds_barrier();
  if (kAhead == 1) {
    for (int l = l0 + 1; l < l1; l += 2) {
      chain_level<1, kUse>(S, X, s_tv, lo, l, l1, base, gs, m, d, daily_slot, a, b);
      if (l + 1 < l1) chain_level<1, kUse>(S, X, s_tv, lo, l + 1, l1, base, gs, m, d, daily_slot, b, a);
    }
  } else {
    for (int l = l0 + 1; l < l1; l += 3) {
      chain_level<2, kUse>(S, X, s_tv, lo, l, l1, base, gs, m, d, daily_slot, a, c);
      if (l + 1 < l1) chain_level<2, kUse>(S, X, s_tv, lo, l + 1, l1, base, gs, m, d, daily_slot, b, a);
      if (l + 2 < l1) chain_level<2, kUse>(S, X, s_tv, lo, l + 2, l1, base, gs, m, d, daily_slot, c, b);
    }
  }
  (void)T;
}

// Wave walk of a routing group.  The levels above level 0 are routed in batches of
// up to 64 cells, one cell per lane, each lane's inputs loaded one batch before
// the batch is routed; transported volumes pass between lanes through LDS.
//  - The leading wide levels (more than 64 cells) are cut into level-aligned
//    batches dealt round-robin to the workgroup's kWaves wavefronts (4 or 8),
//    with an LDS-only barrier after each level.
//  - The narrow rest is routed by wavefront 0 alone in batches of 64 cells taken
//    in device order (by level), so that a batch covers several narrow levels;
//    within a batch the levels run in order, each on the lanes whose cells lie
//    on it.  LDS serves the LDS operations of one wavefront in issue order, so
//    no barrier is needed there.
// A batch's results are stored when the batch is done.  Every batch issues the
// same loads and stores (padding batches route nothing), so that no wait covers
// the loads issued for the next batch.
__device__ inline void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
}

// One batch: cells [b0, bend) (b0 >= bend: a padding batch); `q` holds the
// batch's inputs, `fill` receives those of the batch starting at pnext.
// kWide: a batch of the wide levels, where next_lr / cur_lr (uniform) are the
// batches' lakeres flags: the next batch's suffix is loaded, and this batch's
// lake and reservoir stores issued, only when it is 1.  Otherwise a batch of the
// narrow rest: per-cell record suffix through s_fl, every store issued.
template <bool kWide, bool kUse>
__device__ __forceinline__ void wave_batch(const WgStatic &S, const WgState &X, double *s_tv, int b0, int bend,
                                           int pnext, int ge, int gs, int64_t base, int m, const DayInfo &d,
                                           int daily_slot, const uint8_t *s_fl, int next_lr, int cur_lr,
                                           const ChainSlot &q, ChainSlot &fill) {
  const int lane = threadIdx.x & 63;
  {
    const int pf = pnext + lane < ge ? pnext + lane : gs;
    if (kWide)
      prefetch_slot_batch<kUse>(S, X, base, pf, next_lr != 0, fill);
    else
      prefetch_slot_wave<kUse>(S, X, base, pf, s_fl[pf - gs], fill);
  }
  const int p = b0 + lane;
  const bool have = p < bend;
  ChainOut o = {0., 0., 0., 0., 0., 0., 0., 0.};
  bool run = false;
  if (b0 < bend) {
    const int last = min(63, bend - 1 - b0);
    const int lv_a = __builtin_amdgcn_readfirstlane(q.level);
    const int lv_b = __builtin_amdgcn_readlane(q.level, last);
    ChainRec c;
    slot_record(q, c);
    const StepPre pre = step_pre<kUse>(c);
    for (int l = lv_a; l <= lv_b; l++) {
      if (have && q.level == l) {
        // upstream transported volumes in routing order (routing.cpp:3955-3958);
        // entries past the cell's own count read entry 0 and add +0, which leaves
        // the non-negative sum unchanged.  Past the level's largest count (most
        // levels have at most two upstream cells) nothing is added.
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; u++) t[u] = s_tv[(q.up[u >> 1] >> ((u & 1) * 16)) & 0xffff];
        double up = 0.;
        up += t[0];
        up += (q.nu > 1) ? t[1] : 0.;
        if (__builtin_amdgcn_readfirstlane(q.nu_level) > 2) {
#pragma unroll
          for (int u = 2; u < 8; u++) up += (u < q.nu) ? t[u] : 0.;
        }
        bool slow;
        o = step_fast<kUse>(c, pre, up, slow);
        if (slow) o = chain_step<kUse>(c, up, d);
        run = (q.flags & CFL_CONT) != 0;
        s_tv[p - gs] = run ? o.tv : 0.;
      }
      wave_lds_order();
    }
  }
  const int n = S.n;
  if (cur_lr != 0) {
    store_or_drop(X.glo_lake + base, n, run && (q.flags & CFL_LAKE), p, o.glo_lake);
    store_or_drop(X.res + base, n, run && (q.flags & CFL_RES), p, o.res);
    store_or_drop(X.k_release + base, n, run && (q.flags & CFL_RES), p, o.k_release);
  }
  store_or_drop(X.glo_wetl + base, n, run && (q.flags & CFL_GWET), p, o.glo_wetl);
  store_or_drop(X.gw + base, n, run && (q.flags & CFL_ARID), p, o.gw);
  if (X.pot_lgw) store_or_drop(X.pot_lgw + base, n, run && (q.flags & CFL_ARID), p, o.lgw);
  if (kUse) store_or_drop(X.use_rem + base, n, run, p, o.rem);
  store_or_drop(X.river + base, n, run, p, o.river);
  store_or_drop(X.tv + base, n, run, p, o.tv);
  const double qq = (run && (q.flags & CFL_LDD)) ? o.tv : 0.;
  store_or_drop(X.st_daily + (int64_t(m) * WG_DAILY_SLOTS + daily_slot) * S.n_stations, S.n_stations,
                have && q.station >= 0, q.station, qq);
}

template <int kWaves, bool kUse>
__global__ __launch_bounds__(64 * kWaves) void wg_chain_wave_kernel(WgStatic S, WgState X, WgTables T,
                                                            const int32_t *__restrict__ group_level_off,
                                                            const int32_t *__restrict__ group_first_level,
                                                            const int32_t *__restrict__ wave_wide,
                                                            const int32_t *__restrict__ wave_item_off,
                                                            const WgWaveItem *__restrict__ wave_items,
                                                            const WgClock *__restrict__ clock, int k,
                                                            int daily_slot) {
  extern __shared__ double s_tv[];
  const int g = S.block_group[blockIdx.x];
  if (g < 0) return;
  const int m = blockIdx.y;
  const int n = S.n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // the wavefront, uniform
  const int doy = int((clock->doy0 - 1 + k) % 365) + 1;
  const DayInfo d = day_info(doy);
  const int32_t *lo = group_level_off;
  const int l0 = group_first_level[g], l1 = group_first_level[g + 1];
  const int gs = lo[l0], ge = lo[l1];
  if (l1 - l0 < 2 || ge <= gs) return;  // nothing routed in this kernel
  const int lvl0_end = lo[l0 + 1];
  const int64_t base = int64_t(m) * n;
  const int la = wave_wide[g];  // wide levels l0 + 1 .. l0 + la
  const int pb = lo[l0 + 1 + la];  // first cell of the narrow rest
  // level 0 was routed by the cell kernel: its transported volumes, four loads
  // in flight per thread
  constexpr int kThreads = 64 * kWaves;
  // the chain flags of the group's cells, behind its transported volumes (the
  // launch gives every workgroup 9 bytes of LDS per cell of the largest group);
  // both are loaded together, 16 of each in flight per thread
  uint8_t *s_fl = reinterpret_cast<uint8_t *>(s_tv + (ge - gs));
  constexpr int kFill = 16;
  for (int i0 = gs + tid; i0 < ge; i0 += kFill * kThreads) {
    double v[kFill];
    int8_t f[kFill];
#pragma unroll
    for (int j = 0; j < kFill; j++) {
      const int i = i0 + j * kThreads;
      v[j] = (i < lvl0_end) ? X.tv[base + i] : 0.;
      f[j] = (i < ge) ? S.cflags[i] : int8_t(0);
    }
#pragma unroll
    for (int j = 0; j < kFill; j++) {
      const int i = i0 + j * kThreads;
      if (i < lvl0_end) s_tv[i - gs] = v[j];
      if (i < ge) s_fl[i - gs] = uint8_t(f[j]);
    }
  }
  ChainSlot s0, s1;
  // wide levels: this wavefront's batches in level order; a padding batch (past
  // the list) routes nothing and passes no barrier.  Every wavefront passes
  // exactly la barriers, one after each wide level.  The first batch's loads go
  // out with the fill's.
  const int it0 = la > 0 ? wave_item_off[g * kWaves + w] : 0;
  const int it1 = la > 0 ? wave_item_off[g * kWaves + w + 1] : 0;
  auto item = [&](int i) {
    return (i < it1) ? wave_items[i] : WgWaveItem{ge, ge, 0, 0};
  };
  WgWaveItem ia = item(it0);
  if (la > 0) {
    const int pf = ia.start + lane < ge ? ia.start + lane : gs;
    prefetch_slot_batch<kUse>(S, X, base, pf, ia.lakeres != 0, s0);
  }
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  lds_barrier();
  if (la > 0) {
    int lev = 1;
    for (int i = it0; i < it1; i += 2) {
      const WgWaveItem ib = item(i + 1), ic = item(i + 2);
      while (lev < ia.level) {
        lds_barrier();
        lev++;
      }
      wave_batch<true, kUse>(S, X, s_tv, ia.start, ia.end, ib.start, ge, gs, base, m, d, daily_slot, s_fl, ib.lakeres,
                 ia.lakeres, s0, s1);
      while (lev < ib.level) {
        lds_barrier();
        lev++;
      }
      wave_batch<true, kUse>(S, X, s_tv, ib.start, ib.end, ic.start, ge, gs, base, m, d, daily_slot, s_fl, ic.lakeres,
                 ib.lakeres, s1, s0);
      ia = ic;
    }
    while (lev <= la) {
      lds_barrier();
      lev++;
    }
  }
  if (w != 0 || pb >= ge) return;
  // the narrow rest, wavefront 0 alone
  const int nb = (ge - pb + 127) / 128 * 2;
  {
    const int pa = pb + lane < ge ? pb + lane : gs;
    prefetch_slot_wave<kUse>(S, X, base, pa, s_fl[pa - gs], s0);
  }
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  for (int b = 0; b < nb; b += 2) {
    const int b0 = pb + b * 64;
    wave_batch<false, kUse>(S, X, s_tv, b0, ge, b0 + 64, ge, gs, base, m, d, daily_slot, s_fl, 1, 1, s0, s1);
    wave_batch<false, kUse>(S, X, s_tv, b0 + 64, ge, b0 + 128, ge, gs, base, m, d, daily_slot, s_fl, 1, 1, s1, s0);
  }
  (void)T;
}

// Dataflow walk of a routing group, without a barrier per level.  Each thread owns
// the cells of the group's levels at positions tid, tid + nt, ... (so its cells
// come in level order) and routes each one as soon as the transported volumes of
// all its upstream cells are in LDS; LDS holds a sentinel bit pattern until a
// cell's volume is written.  The unfinished cell of lowest level always has its
// inputs ready and its owner at it, so the walk cannot stall; a spin limit that
// every lane reaches ends the kernel (with an error flag) should that ever fail.
constexpr unsigned long long kTvPending = 0xFFF4A11DDEADBEEFull;  // a NaN no arithmetic produces
constexpr uint32_t kFlowSpinLimit = 1u << 24;

__device__ inline bool flow_next(const int32_t *s_lo, int l1_rel, int nt, int &l, int &p) {
  // advance (l, p) to this thread's next cell: same level + nt, else the next level
  // with a cell at this thread's position (l relative to the group's first level)
  p += nt;
  const int tid = threadIdx.x;
  while (l < l1_rel && p >= s_lo[l + 1]) {
    l++;
    if (l < l1_rel) p = s_lo[l] + tid;
  }
  return l < l1_rel;
}

template <bool kUse>
__global__ __launch_bounds__(256) void wg_chain_flow_kernel(WgStatic S, WgState X, WgTables T,
                                                            const int32_t *__restrict__ group_level_off,
                                                            const int32_t *__restrict__ group_first_level,
                                                            const WgClock *__restrict__ clock, int k,
                                                            int daily_slot) {
  extern __shared__ double s_tv[];
  __shared__ int32_t s_lo[WG_MAX_GROUP_DEPTH + 1];
  const int g = S.block_group[blockIdx.x];
  if (g < 0) return;
  const int m = blockIdx.y;
  const int n = S.n;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int doy = int((clock->doy0 - 1 + k) % 365) + 1;
  const DayInfo d = day_info(doy);
  const int l0 = group_first_level[g], l1 = group_first_level[g + 1];
  const int depth = l1 - l0;
  const int gs = group_level_off[l0], ge = group_level_off[l1];
  const int lvl0_end = group_level_off[l0 + 1];
  const int64_t base = int64_t(m) * n;
  for (int i = tid; i <= depth; i += nt) s_lo[i] = group_level_off[l0 + i];
  volatile unsigned long long *vtv = reinterpret_cast<volatile unsigned long long *>(s_tv);
  for (int i = gs + tid; i < ge; i += nt) {
    double v;
    if (i < lvl0_end)
      v = X.tv[base + i];  // level 0 was routed by the cell kernel
    else
      v = (S.clink[i].x & CFL_CONT) ? __longlong_as_double(kTvPending) : 0.;
    s_tv[i - gs] = v;
  }
  __syncthreads();
  int l = 1, p = s_lo[1] + tid;  // level relative to l0
  while (l < depth && p >= s_lo[l + 1]) {
    l++;
    if (l < depth) p = s_lo[l] + tid;
  }
  bool have = l < depth;
  ChainSlot cur, nxt;
  int nl = l, np = p;
  bool have_nxt = false;
  if (have) {
    prefetch_slot(S, X, base, p, cur);
    have_nxt = flow_next(s_lo, depth, nt, nl, np);
    if (have_nxt) prefetch_slot(S, X, base, np, nxt);
  }
  uint32_t spins = 0;
  while (have) {
    if (++spins > kFlowSpinLimit) {
      X.flow_error[0] = 1;
      break;
    }
    bool ready = true;
    if (cur.flags & CFL_CONT) {
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (u < cur.nu && vtv[(cur.up[u >> 1] >> ((u & 1) * 16)) & 0xffff] == kTvPending) ready = false;
    }
    if (!ready) continue;
    double qq = 0.;
    if (cur.flags & CFL_CONT) {
      double up = 0.;
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (u < cur.nu) up += __longlong_as_double(vtv[(cur.up[u >> 1] >> ((u & 1) * 16)) & 0xffff]);
      ChainRec c;
      slot_record(cur, c);
      const ChainOut o = chain_step<kUse>(c, up, d);
      vtv[p - gs] = __double_as_longlong(o.tv);
      store_chain(X, base, p, cur.flags, o);
      qq = (cur.flags & CFL_LDD) ? o.tv : 0.;
    }
    if (cur.station >= 0)
      X.st_daily[(int64_t(m) * WG_DAILY_SLOTS + daily_slot) * S.n_stations + cur.station] = qq;
    have = have_nxt;
    if (have) {
      cur = nxt;
      l = nl;
      p = np;
      have_nxt = flow_next(s_lo, depth, nt, nl, np);
      if (have_nxt) prefetch_slot(S, X, base, np, nxt);
    }
  }
  (void)T;
}

// Adds the daily station discharge of slots [slot0, slot0 + n_slots) to the running
// sums, day by day in order (the per-day += of routing.cpp:4232-4238).
__global__ void wg_station_reduce(WgState X, int32_t n_stations, int32_t n_members, int slot0, int n_slots) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_stations * n_members) return;
  const int m = i / n_stations, st = i - m * n_stations;
  double s = X.st_sum[i];
  const double *q = X.st_daily + (int64_t(m) * WG_DAILY_SLOTS + slot0) * n_stations + st;
  int d = 0;
  for (; d + 8 <= n_slots; d += 8) {  // eight loads in flight, added in day order
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = q[int64_t(d + j) * n_stations];
#pragma unroll
    for (int j = 0; j < 8; j++) s += v[j];
  }
  for (; d < n_slots; d++) s += q[int64_t(d) * n_stations];
  X.st_sum[i] = s;
}

__global__ void wg_pot_runoff_kernel(WgStatic S, WgState X, int32_t p0, int32_t p1) {
  const int p = p0 + int(blockIdx.x * blockDim.x + threadIdx.x);
  if (p >= p1) return;
  if (!(S.cflags[p] & CFL_CONT)) return;
  add_pot_runoff(S, X, int64_t(blockIdx.y) * S.n, p);
}

// ---- state and outputs between the device order and the reference's ----
// Up to kStageRows rows pass at once through a staging buffer [row][N] of doubles in
// reference order; 32-bit integers and floats travel as doubles, which hold them
// exactly.  The host then copies rows to and from pinned memory in order: a day of
// 2,000 cells with its six output fields read went from 253 to 189 us, against one
// pageable copy and a permutation on the host for each row.
constexpr int kStageRows = 32;
enum RowKind : uint8_t { ROW_F64, ROW_I32, ROW_F32 };
struct StageRows {
  void *row[kStageRows];
  uint8_t kind[kStageRows];
};

// stage[f][ref[p]] = row f of one member at p (ROW_F64 or ROW_I32)
__global__ void wg_rows_out(StageRows rows, const int32_t *__restrict__ ref, int32_t n, double *__restrict__ stage) {
  const int p = int(blockIdx.x * blockDim.x + threadIdx.x), f = blockIdx.y;
  if (p >= n) return;
  const void *r = rows.row[f];
  stage[int64_t(f) * n + ref[p]] =
      rows.kind[f] == ROW_F64 ? static_cast<const double *>(r)[p] : double(static_cast<const int32_t *>(r)[p]);
}

// row f at p = stage[f][ref[p]], for n_members members from the row's
__global__ void wg_rows_in(StageRows rows, const int32_t *__restrict__ ref, int32_t n, int32_t n_members,
                           const double *__restrict__ stage) {
  const int p = int(blockIdx.x * blockDim.x + threadIdx.x), f = blockIdx.y;
  if (p >= n) return;
  const double v = stage[int64_t(f) * n + ref[p]];
  for (int m = 0; m < n_members; m++) {
    const int64_t i = int64_t(m) * n + p;
    if (rows.kind[f] == ROW_F64)
      static_cast<double *>(rows.row[f])[i] = v;
    else if (rows.kind[f] == ROW_I32)
      static_cast<int32_t *>(rows.row[f])[i] = int32_t(v);
    else
      static_cast<float *>(rows.row[f])[i] = float(v);
  }
}

// Sub-cell storages of one member's reference cells c0 to c1 to [cell][channels]
// (channel 0, which the day loop has no copy of, is left alone), and from there to
// n_members members with the flag whether any of a cell's is not exactly zero.
__global__ void wg_snow_out(const WgD2 *__restrict__ snow, const int32_t *__restrict__ ref, int32_t n,
                            int32_t channels, int32_t c0, int32_t c1, double *__restrict__ stage) {
  const int p = int(blockIdx.x * blockDim.x + threadIdx.x), k = blockIdx.y;
  if (p >= n || ref[p] < c0 || ref[p] >= c1) return;
  const WgD2 v = snow[int64_t(k) * n + p];
  double *d = stage + int64_t(ref[p] - c0) * channels + 1 + 2 * k;
  d[0] = v.x;
  d[1] = v.y;
}

__global__ void wg_snow_in(WgD2 *__restrict__ snow, uint8_t *__restrict__ any, const int32_t *__restrict__ ref,
                           int32_t n, int32_t channels, int32_t c0, int32_t c1, int32_t n_members,
                           const double *__restrict__ stage) {
  const int p = int(blockIdx.x * blockDim.x + threadIdx.x);
  if (p >= n || ref[p] < c0 || ref[p] >= c1) return;
  const double *d = stage + int64_t(ref[p] - c0) * channels + 1;
  bool nz = false;
  for (int k = 0; k < WG_DEV_NPAIR; k++) {
    const WgD2 v{d[2 * k], d[2 * k + 1]};
    nz = nz || v.x != 0. || v.y != 0.;
    for (int m = 0; m < n_members; m++) snow[(int64_t(m) * WG_DEV_NPAIR + k) * n + p] = v;
  }
  for (int m = 0; m < n_members; m++) any[int64_t(m) * n + p] = nz ? 1 : 0;
}

// Sets the day clock read by the kernels of a captured block of days; launched
// before each replay so that one graph serves every block of the same length.
__global__ void wg_clock_set(WgClock *clock, int64_t day0, int32_t doy0, int32_t started) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    clock->day0 = day0;
    clock->doy0 = doy0;
    clock->started = started;
  }
}

// Evaluates the shared math functions on the device for a batch of arguments
// (0: wg_exp(x), 1: wg_pow(x, y), 2: sqrt(x), 3: wg_log(x)); used to show that
// the device returns the host's bits.
__global__ void wg_libm_kernel(int fn, int n, const double *__restrict__ x, const double *__restrict__ y,
                               double *__restrict__ out) {
  load_exp2_table();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double r;
  switch (fn) {
    case 0: r = wg_exp(x[i]); break;
    case 1: r = wg_pow(x[i], y[i]); break;
    case 2: r = sqrt(x[i]); break;
    case 3: r = wg_log(x[i]); break;
    default: {
      double sn, cs;
      wg_sincos2pi(x[i], &sn, &cs);
      r = (fn == 4) ? sn : cs;
      break;
    }
  }
  out[i] = r;
}
