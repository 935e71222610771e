// wg_days_kernel.h -- many days of the day loop in one launch: each wavefront keeps
// 64 cells for all days of a block and passes transported volumes to the
// wavefronts downstream through a ring in memory.
//
// Water moves only downstream, so day d of a cell needs day d of the cells above it
// and its own day d - 1, nothing else: upstream wavefronts may run days ahead, and a
// day costs a wavefront its own work instead of the slowest cell's day plus the
// deepest group's walk (the bound of one launch per day and part).
//
// Ring: [slot][member][N] transported volumes of the last ring_slots days, slot =
// (days since the ring was cleared) mod ring_slots.  A volume is never negative, so
// its sign bit says which turn of the ring wrote it: a reader waits until the sign
// is the turn's, and value and flag arrive in one 8-byte access at agent scope (the
// XCDs' L2 caches are not coherent for plain accesses).  A launch covers at most
// ring_slots days, so it never overwrites a volume that it has yet to read.
//
// Wavefronts take the cells in level order over the whole grid, so that one of them
// spans few levels (often one): a level within a wavefront costs a pass of the
// routing step each day, a level between wavefronts only delays the first day.
//
// Progress: a wavefront waits only for cells before its own in level order, never
// for later ones, and each XCD starts a launch's workgroups in index order; so the first
// unfinished wavefront can always run, as long as no other waiting launch holds the
// slots it needs (wg_day_gate.h).  A spin limit ends the launch with an error flag
// should that ever fail, as it might where processes share a GPU.
#ifndef WG_DAYS_KERNEL_H
#define WG_DAYS_KERNEL_H

namespace {

// Per-cell statics and some of the state, kept in LDS, [field][64 lanes] doubles
// behind the exp/log/pow table: read once per launch instead of once per day from
// memory, and out of registers.  Two wavefronts per SIMD hold 256 registers each; the
// kernel is kept within them, because a spill costs a memory round trip a day and
// because this compiler can place a spill's store before the point where a branch's
// lanes rejoin.
enum DayField : int {
  // the same for every member
  DF_M_PREC, DF_ALPHA, DF_PET_MXDY, DF_M_NETRAD, DF_MCWH, DF_SNOWFZ, DF_SNOWMT, DF_GRADNT, DF_MELT, DF_ALBEDO,
  DF_ALBEDO_SNOW, DF_EMIS, DF_LAI, DF_CLASS, DF_GWF, DF_PCRIT, DF_AREA, DF_AREA_M, DF_CF100, DF_FSWB, DF_E_GW,
  DF_INV_KGW, DF_OME_GW, DF_E_SW, DF_K_SW, DF_INV_KSW, DF_OME_SW, DF_RED_EXP, DF_LL, DF_LL100, DF_LL_MAX, DF_LW,
  DF_LW100, DF_LW_MAX, DF_GW, DF_GW_MAX, DF_LENGTH, DF_BOTTOM, DF_VEL_C1, DF_VEL_C2, DF_RW_C0, DF_RW_C1, DF_RW_C2,
  DF_RW_C3, DF_RIVER_MAX, DF_MAX_RAF,
  DF_NEAR,  // WgDaySlot's near_lo and near_hi
  DF_SHARED,
  // a member's own: parameters, and state that a day reads once or few cells have
  DF_SMAX = DF_SHARED, DF_GAMMA, DF_CFA, DF_LAI_PREC, DF_TRANSFER, DF_GLO_LAKE, DF_RES, DF_K_RELEASE, DF_RED_GL,
  DF_RED_RES, DF_RED_RIVER, DF_FRAC_CHANGE,
  DF_TV,  // the day's transported volumes of the wavefront's cells
  DF_ROWS
};
// A workgroup is one wavefront, or two that hold the same cells of two members and
// share the members' common rows (both write them, with the same values).
constexpr int days_lds_bytes(int waves) {
  return waves * WG_EXP2_LDS_BYTES + (DF_SHARED + waves * (DF_ROWS - DF_SHARED)) * 64 * int(sizeof(double));
}
// LDS is given out in steps of 1,280 bytes.  One wavefront's rows take 25 of them, so
// that a CU's 160 KB hold five (with 32,768 bytes only four started, whatever the
// occupancy query says, and the rest of the grid waited for whole launches); two
// members' take 32, so that they hold four workgroups, the eight wavefronts that the
// registers allow.
constexpr int kLdsStep = 1280;
static_assert(days_lds_bytes(1) <= 25 * kLdsStep, "five wavefronts per CU");
static_assert(days_lds_bytes(2) <= 32 * kLdsStep, "four workgroups of two wavefronts per CU");

// bits of DF_GWF's second word, whose upper half holds G_Rgmax
enum { DB_ARID = 1, DB_CUT = 2, DB_LDD = 4, DB_CONT = 8, DB_LAKE = 16, DB_RES = 32, DB_FULL_LAKE = 64 };

struct WordPair {
  int32_t a, b;
};

constexpr int kDaysSpinLimit = 1 << 22;
constexpr int kEarly = 3;  // upstream cells whose volumes are loaded ahead (few cells have more)

}  // namespace

// The kernel's arguments, read where they are used: each DAYS_ARGS makes the compiler
// load those that follow anew (scalar loads).  Held in scalar registers from the
// start they would take ten times what there is, spilled lane by lane (a sixth of
// the vector instructions of a day).  About 160 scalar spills are left, to lanes of
// vector registers: lane masks and row addresses that live across the day loop.
struct DaysArgs {
  WgStatic stat;
  WgState state;
  WgTables tables;
  const float *forcing;
  const WgDayWave *waves;
  const WgDaySlot *slots;
  const uint8_t *ranks;
  unsigned long long *ring;
  int64_t fday0;
  int32_t ring_slots, ring_slot0, ring_turn;  // the first day's slot, and its turn's parity
  int32_t doy0, started0, days, slot0;
};
typedef const __attribute__((address_space(4))) DaysArgs *DaysArgsPtr;
#define DAYS_ARGS(A, S, X)                                              \
  DaysArgsPtr A##_ = (DaysArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(); \
  asm volatile("" : "+s"(A##_));                                        \
  const DaysArgs &A = *(const DaysArgs *)A##_;                          \
  const WgStatic &S = A.stat;                                              \
  const WgState &X = A.state;                                               \
  (void)S;                                                              \
  (void)X

namespace {

__device__ __forceinline__ int days_doy(const DaysArgs &A, int k) { return int((A.doy0 - 1 + k) % 365) + 1; }
__device__ __forceinline__ DayInfo days_info(const DaysArgs &A, int k) { return day_info(days_doy(A, k)); }

// Upstream cell u's volume of the day, as it stands in the ring.
__device__ __forceinline__ unsigned long long days_volume(unsigned long long *row, int group, const WgChainLink &link,
                                                          int u) {
  return __hip_atomic_load(&at(row, uint32_t(group) + uint16_t(link.up[u])), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// The member's row of day k in the ring, and the sign bit of its turn.
__device__ __forceinline__ unsigned long long *days_ring_row(const DaysArgs &A, int k, int64_t o,
                                                             unsigned long long &sign) {
  const uint32_t slots = uint32_t(A.ring_slots), at0 = uint32_t(A.ring_slot0) + uint32_t(k);
  const bool wrapped = at0 >= slots;  // at most once in a launch
  sign = (wrapped != (A.ring_turn != 0)) ? 0ull : 0x8000000000000000ull;
  return A.ring + int64_t(wrapped ? at0 - slots : at0) * A.stat.n_members * A.stat.n + o;
}

__device__ __forceinline__ double *days_station_row(const DaysArgs &A, int k, int m) {
  return A.state.st_daily + (int64_t(m) * WG_DAILY_SLOTS + A.slot0 + k) * A.stat.n_stations;
}

}  // namespace

template <bool kUse, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 2) void wg_days_kernel(DaysArgs) {
  load_exp2_table();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = blockIdx.y * kWaves + wave;
  DAYS_ARGS(A0, S0, X0);
  if (kWaves > 1 && m >= S0.n_members) return;
  const WgDayWave wv = A0.waves[blockIdx.x];
  const WgDaySlot slot = A0.slots[blockIdx.x * 64 + lane];
  if (slot.cell < 0) return;
  const uint32_t p = uint32_t(slot.cell);
  const int n = S0.n;
  const int64_t o = int64_t(m) * n;  // the member's rows
  double *Fs = wg_lds + kWaves * WG_EXP2_LDS_BYTES / sizeof(double) + lane;
  double *Fm = Fs + wave * (DF_ROWS - DF_SHARED) * 64;
  auto row = [&](int f) -> double & { return f < DF_SHARED ? Fs[f * 64] : Fm[f * 64]; };
  auto fld = [&](int f) -> double { return row(f); };

  const WgChainLink link = load_link(S0, p);
  const int rank = A0.ranks[blockIdx.x * 64 + lane];
  row(DF_NEAR) = __builtin_bit_cast(double, WordPair{int32_t(slot.near_lo), int32_t(slot.near_hi)});
  int bits = 0;
  {
    DayStatA a;
    DayStatB b;
    DayStatEnd e;
    load_stat_a(S0, A0.tables, p, a);
    load_stat_b(S0, X0, o, p, b);
    load_stat_end(S0, p, e);
    const WgChainStatic cs = load_cstat(S0, p);
    bits = (b.arid ? DB_ARID : 0) | (b.recharge_cut ? DB_CUT : 0) | (b.ldd >= 0 ? DB_LDD : 0) |
           (e.contcell ? DB_CONT : 0) | (e.lake_area > 0. ? DB_LAKE : 0) | (e.reservoir_area > 0. ? DB_RES : 0) |
           (e.f_glo_lake == 1. ? DB_FULL_LAKE : 0) | int(uint32_t(uint16_t(at(S0.rgmax, p))) << 16);
    row(DF_M_PREC) = a.m_prec;
    row(DF_ALPHA) = a.alpha;
    row(DF_PET_MXDY) = a.pet_mxdy;
    row(DF_M_NETRAD) = a.m_netrad;
    row(DF_MCWH) = a.mcwh;
    row(DF_SNOWFZ) = a.t_snowfz;
    row(DF_SNOWMT) = a.t_snowmt;
    row(DF_GRADNT) = a.t_gradnt;
    row(DF_MELT) = a.melt_factor;
    row(DF_ALBEDO) = a.albedo;
    row(DF_ALBEDO_SNOW) = a.albedo_snow;
    row(DF_EMIS) = a.emis;
    row(DF_LAI) = __builtin_bit_cast(double, WordPair{__builtin_bit_cast(int32_t, float(a.lmin)),
                                                         __builtin_bit_cast(int32_t, float(a.lmax))});
    row(DF_CLASS) = __builtin_bit_cast(double, WordPair{a.initial_days, a.lct | (a.elev0 << 8)});
    row(DF_SMAX) = __builtin_bit_cast(double, WordPair{__builtin_bit_cast(int32_t, b.smax),
                                                          __builtin_bit_cast(int32_t, b.built_up)});
    row(DF_GWF) = __builtin_bit_cast(double, WordPair{__builtin_bit_cast(int32_t, b.gw_factor), bits});
    row(DF_GAMMA) = b.gamma;
    row(DF_CFA) = b.cfa;
    row(DF_PCRIT) = b.pcritgwa;
    row(DF_AREA) = b.area;
    row(DF_AREA_M) = b.area_m;
    row(DF_CF100) = b.cf100;
    row(DF_FSWB) = b.fswb_catchment;
    row(DF_E_GW) = b.e_gw;
    row(DF_INV_KGW) = cs.inv_kgw;
    row(DF_OME_GW) = cs.ome_gw;
    row(DF_E_SW) = b.e_sw;
    row(DF_K_SW) = b.k_sw;
    row(DF_INV_KSW) = cs.inv_ksw;
    row(DF_OME_SW) = cs.ome_sw;
    row(DF_RED_EXP) = b.red_exp;
    row(DF_LL) = b.loc_lake;
    row(DF_LL100) = b.ll100;
    row(DF_LL_MAX) = b.ll_max;
    row(DF_LW) = b.loc_wetland;
    row(DF_LW100) = b.lw100;
    row(DF_LW_MAX) = b.lw_max;
    row(DF_GW) = b.glo_wetland;
    row(DF_GW_MAX) = b.gw_max;
    row(DF_LENGTH) = b.river_length;
    row(DF_BOTTOM) = b.bottom;
    row(DF_VEL_C1) = b.vel_c1;
    row(DF_VEL_C2) = b.vel_c2;
    row(DF_RW_C0) = e.rw_c0;
    row(DF_RW_C1) = e.rw_c1;
    row(DF_RW_C2) = e.rw_c2;
    row(DF_RW_C3) = e.rw_c3;
    row(DF_RIVER_MAX) = e.river_stor_max;
    row(DF_MAX_RAF) = e.max_raf;
    row(DF_TV) = 0.;
  }
  const bool cont = (bits & DB_CONT) != 0;
  // upstream cells: bit u of ext when upstream cell u belongs to an earlier wavefront
  uint32_t ext = 0;
  if (cont) {
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (u < link.nu && ((u < 4 ? slot.near_lo : slot.near_hi) >> (8 * (u & 3)) & 0xffu) == 0xffu) ext |= 1u << u;
  }

  CellState s;
  load_state_a(X0, o, p, s);
  load_state_b(X0, o, p, s);
  load_state_end(X0, o, p, s);
  s.laf_prev = at(X0.laf_prev + o, p);
  s.red_gl = at(X0.red_gl + o, p);
  s.red_res = at(X0.red_res + o, p);
  row(DF_LAI_PREC) = s.lai_precsum;
  row(DF_TRANSFER) = s.transfer;
  row(DF_GLO_LAKE) = s.glo_lake;
  row(DF_RES) = s.res;
  row(DF_K_RELEASE) = s.k_release;
  row(DF_RED_GL) = s.red_gl;
  row(DF_RED_RES) = s.red_res;
  row(DF_RED_RIVER) = s.red_river;
  row(DF_FRAC_CHANGE) = s.river_frac_change;
  const ElevRange er = load_elev_range(S0, p);
  const float *fd = A0.forcing + A0.fday0 * 4 * int64_t(n);
  const int days = A0.days;
  float f0 = 0.f, f1 = 0.f, f2 = 0.f, f3 = 0.f;
  if (!kUse) {
    f0 = at(fd, p);
    f1 = at(fd + n, p);
    f2 = at(fd + 2 * int64_t(n), p);
    f3 = at(fd + 3 * int64_t(n), p);
  }

#pragma unroll 1
  for (int k = 0; k < days; k++) {
    double rem = 0.;
    if (!cont) {
      DAYS_ARGS(A, S, X);
      unsigned long long sign;
      unsigned long long *rrow = days_ring_row(A, k, o, sign);
      // calcNewDay and routing run for continental cells only (integrateWGHM.cpp:770,
      // routing.cpp:1876); other cells keep a zero transported volume.
      __hip_atomic_store(&at(rrow, p), sign, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (link.station >= 0) days_station_row(A, k, m)[link.station] = 0.;
    } else {
      // the next day's forcing is loaded a day ahead (with water use there is no
      // register to hold it)
      float tf = kUse ? at(fd, p) : f0, pf = kUse ? at(fd + n, p) : f1;
      const float swf = kUse ? at(fd + 2 * int64_t(n), p) : f2, lwf = kUse ? at(fd + 3 * int64_t(n), p) : f3;
      if (kUse) fd += 4 * int64_t(n);
      if (!kUse && k + 1 < days) {
        fd += 4 * int64_t(n);
        f0 = at(fd, p);
        f1 = at(fd + n, p);
        f2 = at(fd + 2 * int64_t(n), p);
        f3 = at(fd + 3 * int64_t(n), p);
      }
      bool started;
      {
        DAYS_ARGS(A, S, X);
        if (X.perturb) perturb_forcing(S, X, m, p, A.fday0 + k, tf, pf);
        started = A.started0 || k > 0;
      }
      const double laf_prev = started ? s.laf_prev : s.laf;  // daily.cpp:159-169
      DayFlux v;
      {
        DayStatA a;
        a.m_prec = fld(DF_M_PREC);
        a.alpha = fld(DF_ALPHA);
        a.pet_mxdy = 0.;
        a.m_netrad = fld(DF_M_NETRAD);
        a.mcwh = fld(DF_MCWH);
        a.t_snowfz = fld(DF_SNOWFZ);
        a.t_snowmt = fld(DF_SNOWMT);
        a.t_gradnt = fld(DF_GRADNT);
        a.melt_factor = fld(DF_MELT);
        a.albedo = fld(DF_ALBEDO);
        a.albedo_snow = fld(DF_ALBEDO_SNOW);
        a.emis = fld(DF_EMIS);
        const WordPair lai = __builtin_bit_cast(WordPair, fld(DF_LAI)), cl = __builtin_bit_cast(WordPair, fld(DF_CLASS));
        a.lmin = __builtin_bit_cast(float, lai.a);
        a.lmax = __builtin_bit_cast(float, lai.b);
        a.initial_days = cl.a;
        a.lct = cl.b & 0xff;
        a.elev0 = cl.b >> 8;
        a.arid = (bits & DB_ARID) != 0;
        s.lai_precsum = fld(DF_LAI_PREC);
        s.transfer = fld(DF_TRANSFER);
        day_pet_canopy(a, s, v, tf, pf, swf, lwf, laf_prev);
        row(DF_LAI_PREC) = s.lai_precsum;
        DAYS_ARGS(A, S, X);
        WgD2 *sub = X.snow2 + o * WG_DEV_NPAIR;
        if (s.laf <= 0.) day_snow_no_land(s, v, sub, p, n);
        row(DF_TRANSFER) = s.transfer;
        // with land, or a fraction that is not a number (as wg_cell_kernel's else)
        if (!(s.laf <= 0.)) day_snow<5, true>(a, s, v, laf_prev, er, sub, S.elev_pairs, p, n);
      }
      // Transported volumes of upstream cells in earlier wavefronts: they are there
      // already unless this wavefront has caught up, so those of the first kEarly
      // upstream cells are loaded before soil and local routing and looked at after.
      DAYS_ARGS(A, S, X);
      unsigned long long sign;
      unsigned long long *rrow = days_ring_row(A, k, o, sign);
      unsigned long long t[8];
#pragma unroll
      for (int u = 0; u < kEarly; u++)
        if (u < wv.nu && (ext >> u & 1)) t[u] = days_volume(rrow, slot.group, link, u);
      ChainRec c;
      {
        DayStatB b;
        const WordPair sm = __builtin_bit_cast(WordPair, fld(DF_SMAX)), gf = __builtin_bit_cast(WordPair, fld(DF_GWF));
        b.smax = __builtin_bit_cast(float, sm.a);
        b.built_up = __builtin_bit_cast(float, sm.b);
        b.gw_factor = __builtin_bit_cast(float, gf.a);
        b.gamma = fld(DF_GAMMA);
        b.cfa = fld(DF_CFA);
        b.pet_mxdy = fld(DF_PET_MXDY);
        b.t_snowfz = fld(DF_SNOWFZ);
        b.pcritgwa = fld(DF_PCRIT);
        b.rgmax = (gf.b >> 16) / 100.;  // G_Rgmax, an int16
        b.recharge_cut = (bits & DB_CUT) != 0;
        b.arid = (bits & DB_ARID) != 0;
        b.ldd = (bits & DB_LDD) ? 0 : -1;
        s.transfer = fld(DF_TRANSFER);
        day_soil(b, s, v, laf_prev);
        row(DF_TRANSFER) = s.transfer;
        if (k == days - 1) {
          DAYS_ARGS(A, S, X);
          at(X.d_surf + o, p) = v.surf_runoff;
          at(X.d_recharge + o, p) = v.recharge;
          at(X.d_ow_pet + o, p) = v.ow_pet;
          at(X.d_aet + o, p) = v.aet;
          at(X.d_prec + o, p) = v.prec;
        }
        DAYS_ARGS(A, S, X);
        double use_desired = 0., use_nag = 0.;
        int64_t use_t = 0;
        if (kUse) use_t = day_use(S, X, o, p, A.fday0 + k, days_info(A, k).month, use_desired, use_nag);
        b.area = fld(DF_AREA);
        b.area_m = fld(DF_AREA_M);
        b.cf100 = fld(DF_CF100);
        b.fswb_catchment = fld(DF_FSWB);
        b.e_gw = fld(DF_E_GW);
        b.inv_kgw = fld(DF_INV_KGW);
        b.ome_gw = fld(DF_OME_GW);
        b.e_sw = fld(DF_E_SW);
        b.k_sw = fld(DF_K_SW);
        b.red_exp = fld(DF_RED_EXP);
        b.loc_lake = fld(DF_LL);
        b.ll100 = fld(DF_LL100);
        b.ll_max = fld(DF_LL_MAX);
        b.loc_wetland = fld(DF_LW);
        b.lw100 = fld(DF_LW100);
        b.lw_max = fld(DF_LW_MAX);
        b.glo_wetland = fld(DF_GW);
        b.gw100 = b.glo_wetland / 100.;
        b.gw_max = fld(DF_GW_MAX);
        b.river_length = fld(DF_LENGTH);
        b.bottom = fld(DF_BOTTOM);
        b.vel_b4 = -b.bottom / 4.0;
        b.vel_b16 = b.bottom * b.bottom / 16.0;
        b.vel_c1 = fld(DF_VEL_C1);
        b.vel_c2 = fld(DF_VEL_C2);
        // global lakes and reservoirs (one cell in a hundred) read their statics here
        DayStatLake lake{0., 0., 0., 0., 0., 0.};
        s.glo_lake = s.red_gl = s.res = s.red_res = s.k_release = 0.;
        if ((bits & (DB_LAKE | DB_RES)) || (link.flags & (CFL_LAKE | CFL_RES))) {
          load_stat_lake(S, p, lake);
          s.glo_lake = fld(DF_GLO_LAKE);
          s.red_gl = fld(DF_RED_GL);
          s.res = fld(DF_RES);
          s.red_res = fld(DF_RED_RES);
          s.k_release = fld(DF_K_RELEASE);
          if (kUse) lake.prov_rel = at(S.use_provrel + use_t, p);
        }
        c.inv_ksw = fld(DF_INV_KSW);
        c.ome_sw = fld(DF_OME_SW);
        c.inv_kgw = b.inv_kgw;
        c.ome_gw = b.ome_gw;
        c.area = b.area;
        c.cf100 = b.cf100;
        c.flags = link.flags;
        PotTerms pot;
        day_local_routing<kUse>(b, lake, s, v, use_desired, use_nag, c, pot);
        if (X.pot_base) {
          at(X.pot_base + o, p) = pot.base;
          at(X.pot_ow + o, p) = pot.ow;
        }
      }
      // wait for the volumes that were not there yet, and load those past the first
      // kEarly upstream cells
      int spins = 0;
      for (;;) {
        bool ready = true;
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (u < wv.nu && (ext >> u & 1)) {
            if (u >= kEarly || spins > 0) t[u] = days_volume(rrow, slot.group, link, u);
            ready = ready && ((t[u] ^ sign) >> 63) == 0;
          }
        if (__builtin_amdgcn_ballot_w64(!ready) == 0) break;
        if (++spins >= kDaysSpinLimit ||
            ((spins & 1023) == 0 &&
             __hip_atomic_load(X.flow_error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          __hip_atomic_store(X.flow_error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(X.flow_error_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          return;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      const StepPre pre = step_pre<kUse>(c);
      ChainOut r = {0., 0., 0., 0., 0., 0., 0., 0., 0.};
      for (int pass = 0; pass < wv.passes; pass++) {
        if (rank == pass) {
          // gather in routing order (the serial += of routing.cpp:3955-3958)
          double up = 0.;
          const WordPair lanes = __builtin_bit_cast(WordPair, fld(DF_NEAR));
#pragma unroll
          for (int u = 0; u < 8; u++)
            if (u < wv.nu) {
              const int near_lane = int(uint32_t(u < 4 ? lanes.a : lanes.b) >> (8 * (u & 3))) & 63;
              const double near = (&row(DF_TV))[near_lane - lane];
              const double far = __builtin_bit_cast(double, t[u] & 0x7fffffffffffffffull);
              const double q = (ext >> u & 1) ? far : near;
              up += (u < link.nu) ? q : 0.;
            }
          bool slow;
          r = step_fast<kUse>(c, pre, up, slow);
          if (slow) {
            DAYS_ARGS(A, S, X);
            r = chain_step<kUse>(c, up, days_info(A, k));
          }
          const unsigned long long w = __builtin_bit_cast(unsigned long long, r.tv) & 0x7fffffffffffffffull;
          __hip_atomic_store(&at(rrow, p), w | sign, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          row(DF_TV) = r.tv;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      }
      if (c.flags & CFL_LAKE) row(DF_GLO_LAKE) = r.glo_lake;
      if (c.flags & CFL_RES) {
        row(DF_RES) = r.res;
        row(DF_K_RELEASE) = r.k_release;
      }
      if (c.flags & CFL_GWET) s.glo_wetl = r.glo_wetl;
      if (c.flags & CFL_ARID) s.gw = r.gw;
      s.river = r.river;
      rem = r.rem;
      {
        DAYS_ARGS(B, SB, XB);
        if (link.station >= 0) days_station_row(B, k, m)[link.station] = (c.flags & CFL_LDD) ? r.tv : 0.;
        if (k == days - 1) at(XB.tv + o, p) = r.tv;
        if (XB.pot_acc) {
          if (c.flags & CFL_ARID) at(XB.pot_lgw + o, p) = r.lgw;
          add_pot_runoff(SB, XB, o, p);
        }
      }
    }
    {
      DayStatEnd e;
      e.red_exp = fld(DF_RED_EXP);
      e.area = fld(DF_AREA);
      e.river_length = fld(DF_LENGTH);
      e.rw_c0 = fld(DF_RW_C0);
      e.rw_c1 = fld(DF_RW_C1);
      e.rw_c2 = fld(DF_RW_C2);
      e.rw_c3 = fld(DF_RW_C3);
      e.river_stor_max = fld(DF_RIVER_MAX);
      e.max_raf = fld(DF_MAX_RAF);
      e.f_glo_lake = (bits & DB_FULL_LAKE) ? 1. : 0.;
      e.loc_lake = fld(DF_LL);
      e.loc_wetland = fld(DF_LW);
      e.glo_wetland = fld(DF_GW);
      e.gw_max = fld(DF_GW_MAX);
      e.lake_area = 0.;
      e.lake_max = 0.;
      e.reservoir_area = 0.;
      e.stor_cap = 0.;
      if (bits & (DB_LAKE | DB_RES)) {
        DAYS_ARGS(A, S, X);
        e.lake_area = at(S.lake_area, p);
        e.lake_max = e.lake_area * at(S.lake_depth, p);
        e.reservoir_area = at(S.reservoir_area, p);
        e.stor_cap = at(S.stor_cap, p);
        s.glo_lake = fld(DF_GLO_LAKE);
        s.red_gl = fld(DF_RED_GL);
        s.res = fld(DF_RES);
        s.red_res = fld(DF_RED_RES);
      }
      e.contcell = cont;
      s.red_river = fld(DF_RED_RIVER);
      s.river_frac_change = fld(DF_FRAC_CHANGE);
      if (kUse && cont) {
        DAYS_ARGS(A, S, X);
        const int fin_ym = int((A.fday0 + k - S.use_day0) / 365) * 12 + days_info(A, k).month;
        day_end_use(S, X.use + o, p, s, rem, e.loc_lake, fld(DF_LL_MAX), e.red_exp, fin_ym,
                    days_doy(A, k) == 365);
      }
      day_end(e, s);
      row(DF_RED_RIVER) = s.red_river;
      row(DF_FRAC_CHANGE) = s.river_frac_change;
      if (bits & (DB_LAKE | DB_RES)) {
        row(DF_RED_GL) = s.red_gl;
        row(DF_RED_RES) = s.red_res;
      }
    }
  }

  DAYS_ARGS(A, S, X);
  at(X.canopy + o, p) = s.canopy;
  at(X.soil + o, p) = s.soil;
  at(X.snow + o, p) = s.snow;
  at(X.transfer + o, p) = fld(DF_TRANSFER);
  at(X.lai_precsum + o, p) = fld(DF_LAI_PREC);
  at(X.lai_days + o, p) = s.lai_days;
  at(X.lai_status + o, p) = s.lai_status;
  at(X.snow_any + o, p) = s.snow_any ? 1 : 0;
  at(X.gw + o, p) = s.gw;
  at(X.loc_lake + o, p) = s.loc_lake;
  at(X.loc_wetl + o, p) = s.loc_wetl;
  at(X.glo_lake + o, p) = fld(DF_GLO_LAKE);
  at(X.glo_wetl + o, p) = s.glo_wetl;
  at(X.res + o, p) = fld(DF_RES);
  at(X.river + o, p) = s.river;
  at(X.red_ll + o, p) = s.red_ll;
  at(X.red_lw + o, p) = s.red_lw;
  at(X.red_gl + o, p) = fld(DF_RED_GL);
  at(X.red_gw + o, p) = s.red_gw;
  at(X.red_res + o, p) = fld(DF_RED_RES);
  at(X.red_river + o, p) = fld(DF_RED_RIVER);
  at(X.river_frac_next + o, p) = s.river_frac_next;
  at(X.river_frac_change + o, p) = fld(DF_FRAC_CHANGE);
  at(X.fswb_next + o, p) = s.fswb_next;
  at(X.laf + o, p) = s.laf;
  at(X.laf_prev + o, p) = s.laf_prev;
  at(X.k_release + o, p) = fld(DF_K_RELEASE);
}

#endif  // WG_DAYS_KERNEL_H
