// wg_cell_day.h -- one cell's day without upstream water: PET, LAI, canopy, snow,
// soil, the part of the routing loop that reads no upstream water, and the day's
// end (reduction factors, river width, surface-water and land area fractions).
//
// Functions from registers to registers: the kernels load the cell's statics and
// state, call them in order and store what they changed.  Terms that are constant
// per cell (maximum storages, exponents, unit factors) are inputs, computed with
// the reference's operations on the same operands, so that a kernel that keeps a
// cell for many days evaluates them once.
#ifndef WG_CELL_DAY_H
#define WG_CELL_DAY_H

// updateNetAbstractionGW, routing.cpp:5503-5572: the day's net abstraction from
// groundwater, with the return flows of irrigation from surface water reduced
// when the last day's surface-water use went unsatisfied (G_dailyRemainingUse > 0)
// or given back when a delayed use was satisfied (< 0).  U points at the
// member's first water-use field, us is the stride between fields.
__device__ inline double update_net_abstraction_gw(double *U, int64_t us, uint32_t p, double frgi, double nug) {
  double &dru = at(U + WG_USE_DAILY_REMAINING * us, p), &ui = at(U + WG_USE_UNSAT_IRRIG * us, p);
  double &uo = at(U + WG_USE_UNSAT_OTHER * us, p), &rrf = at(U + WG_USE_REDUCED_RETURN * us, p);
  const double wu = at(U + WG_USE_WITHDRAWAL_IRRIG * us, p), cu = at(U + WG_USE_CONSUMPTIVE_IRRIG * us, p);
  if (dru > 1.e-12) {
    if (wu > 0.) {
      const double eff = cu / wu;
      const double factor = 1 - (1 - frgi) * (1 - eff);
      double WUsiNew = 1 / factor * (wu * factor - dru);
      if (WUsiNew < 0.) {
        WUsiNew = 0.;
        ui += wu * factor;
        uo += dru - (wu * factor);
      } else {
        ui += dru;
      }
      const double returnflowChange = (frgi * (1 - eff) * (WUsiNew - wu));
      rrf += returnflowChange;
      dru = 0.;
      return nug - returnflowChange;
    }
    uo += dru;
    return nug;
  }
  if (dru < -1.e-12) {
    double fromIrrig = dru + uo;
    if (fromIrrig < 0.) {
      uo = 0.;
    } else {
      uo += dru;
      dru = 0.;
      return nug;
    }
    if (ui == 0.) {
      dru = 0.;
      return nug;
    }
    double ratio = (fromIrrig / ui);
    if (ratio < -1.) {
      ratio = -1.;
      fromIrrig = ui * -1.;
    }
    const double returnflowChange = (ratio * rrf);
    ui += fromIrrig;
    rrf += returnflowChange;
    dru = 0.;
    return nug - returnflowChange;
  }
  return nug;
}

// annualWaterUsePostProcessing, routing.cpp:5257-5296, for one cell
__device__ inline void water_use_year_end(double *U, int64_t us, uint32_t p) {
  double &tu = at(U + WG_USE_TOTAL_UNSAT * us, p), &ui = at(U + WG_USE_UNSAT_IRRIG * us, p);
  double &uo = at(U + WG_USE_UNSAT_OTHER * us, p), &rrf = at(U + WG_USE_REDUCED_RETURN * us, p);
  double &tu_py = at(U + WG_USE_UNSAT_PREV_YEAR * us, p), &ui_py = at(U + WG_USE_UNSAT_IRRIG_PREV_YEAR * us, p);
  double &uo_py = at(U + WG_USE_UNSAT_OTHER_PREV_YEAR * us, p), &rrf_py = at(U + WG_USE_REDUCED_RETURN_PREV_YEAR * us, p);
  if (tu < tu_py) {
    tu_py = tu;
    ui_py = ui;
    uo_py = uo;
    rrf_py = rrf;
    ui = 0.;
    uo = 0.;
    rrf = 0.;
    tu = 0.;
  } else {
    tu -= tu_py;
    ui -= ui_py;
    uo -= uo_py;
    rrf -= rrf_py;
    if ((ui + uo) < 0) {
      ui = 0;
      uo = 0;
      rrf = 0;
    } else if (uo < 0) {
      ui += uo;
      uo = 0;
    } else if (ui < 0) {
      uo += ui;
      ui = 0;
      rrf = 0;
    }
    if (rrf > 0) {
      rrf = 0;
      ui = 0;
    }
  }
}

// routing.cpp:7309-7341 getNewRiverVelocity
// c1 = 1. / (mult * rough) and c2 = pow(slope, 0.5) are per-cell constants computed
// on the host with the same operations, b4 = -bottom / 4 and b16 = bottom * bottom /
// 16 by the caller, so the result is the reference's.
__device__ inline double new_river_velocity(double c1, double c2, double bottom, double b4, double b16, double stor,
                                            double length) {
  const double csa = (stor / length) * 1000000.;
  const double depth = b4 + sqrt(b16 + 0.5 * csa);
  const double wp = bottom + 2.0 * depth * sqrt(5.0);
  const double hr = csa / wp;
  double v = c1 * wg_pow(hr, (2. / 3.)) * c2;
  v = v * 86.4;
  return (v < 0.00001) ? 0.00001 : v;
}

// LAI state machine, lai.cpp:179-293
__device__ inline double lai_day(int &days, int init_days, int &status, int lct, bool arid, double lmin,
                                 double lmax, double &precsum, double prec, bool growing) {
  if (growing) {
    if (status == 0) {
      if (days >= init_days) {
        days++;
        precsum += prec;
        if (precsum > 40.) {
          if (days >= init_days + 30) {
            days = init_days + 30;
            status = 1;
          }
          return (lmin + (lmax - lmin) * (days - init_days) / 30.);
        }
        days = init_days;
        return lmin;
      }
      days++;
      precsum += prec;
      return lmin;
    }
    if (days <= 30) {
      days--;
      if (lct <= 2) status = 0;
      if (days <= 0) {
        days = 0;
        status = 0;
        precsum = 0.;
      }
      return (lmax - (lmax - lmin) * (30 - days) / 30.);
    }
    if (arid && (prec < 0.5))
      days--;
    else
      days = 30 + init_days;
    return lmax;
  }
  if (status == 0) {
    if (days > init_days) {
      days++;
      precsum += prec;
      if (precsum > 40.) {
        if (days >= init_days + 30) {
          days = init_days + 30;
          status = 1;
        }
        return (lmin + (lmax - lmin) * (days - init_days) / 30.);
      }
      days = init_days;
      return lmin;
    }
    precsum += prec;
    return lmin;
  }
  if (days <= 30) {
    days--;
    if (days <= 0) {
      days = 0;
      status = 0;
      precsum = 0.;
    }
    return (lmax - (lmax - lmin) * (30 - days) / 30.);
  }
  days--;
  return lmax;
}

// ---- one elevation sub-cell of the snow loop, daily.cpp:920-1044 ----

struct SnowDay {
  double tempC, gradnt, scale_num, laf, prec_to_soil, soil_pet, snowfz, snowmt, melt_factor;
  double inv_laf;   // 1 / laf, correctly rounded
  int elev0;
  // melt_factor > 0; any other takes the full step (0 too: an infinite temperature
  // times it is a melt of NaN)
  bool melt_ok;
};

struct SnowAcc {
  double snow_sum, eff, evapo, change, temp_max;
  int thresh;
};

// Updates one sub-cell storage s and the cell's running sums in sub-cell order
// (daily.cpp:920-1044); temp_elev is the sub-cell temperature T - (z_e - z0) gradnt
// and melt_factor = M_DEGDAY_F * ddf_lct (daily.cpp:1013).  The reference's branches
// are selects here: every operation is the reference's, on the same operands, and
// a branch not taken adds +0 to a sum, which leaves it unchanged (the sums start at
// +0 and never hold -0).  Without branches the two sub-cells of a pair are
// independent chains that the compiler interleaves.
__device__ inline double snow_subcell(double s, double temp_elev, int elev_e, bool first, const SnowDay &d,
                                      SnowAcc &a) {
  {
    // s * scale_num / laf with the reused reciprocal: q0 = x (1/laf), one exact
    // residual and one correction give the correctly rounded quotient (Markstein's
    // theorem for a correctly rounded reciprocal; tests/test_division.py compares
    // it with the division on random operands).  An infinite or NaN x is its own quotient by the
    // finite positive laf.  (The quotient of a finite x overflows only for
    // x > 1e292 mm, since a positive land area fraction is at least about 1e-16.)
    const double x = s * d.scale_num;
    const double q0 = x * d.inv_laf;
    const double q = fma(fma(-q0, d.laf, x), d.inv_laf, q0);
    s = (fabs(x) <= 1.7976931348623157e308) ? q : x;
  }
  s = (fabs(s) <= kMinStorVol) ? 0. : s;
  const double init_s = s;
  // threshold elevation above 1000 mm of storage (daily.cpp:958-976)
  const bool big = s > 1000.;
  const bool use_thresh = big && a.thresh > 0;
  const double temp_thresh = d.tempC - ((a.thresh - d.elev0) * d.gradnt);
  a.thresh = (big && a.thresh == 0) ? elev_e : a.thresh;
  temp_elev = use_thresh ? temp_thresh : temp_elev;
  // snowfall and sublimation below the freezing temperature, rain above it
  const bool freeze = temp_elev <= d.snowfz;
  const double s_fall = s + d.prec_to_soil;
  const bool keeps = s_fall > d.soil_pet;
  const double s_subl = s_fall - d.soil_pet;
  a.evapo += freeze ? (keeps ? d.soil_pet : s_fall) : 0.;
  s = freeze ? (keeps ? s_subl : 0.) : s;
  const double eff_before = freeze ? 0. : d.prec_to_soil;
  // degree-day melt
  const bool melts = (temp_elev > d.snowmt) && !(s < 0.);
  const double melt_pot = d.melt_factor * (temp_elev - d.snowmt);
  const bool all = melt_pot > s;
  const double s_left = s - melt_pot;
  const double snowmelt_elev = melts ? (all ? s : melt_pot) : 0.;
  s = melts ? (all ? 0. : s_left) : s;
  const double eff_elev = eff_before + snowmelt_elev;
  a.change += s - init_s;
  if (first) a.temp_max = temp_elev;
  a.snow_sum += s;
  a.eff += eff_elev;
  return s;
}

// Statics of PET, LAI, canopy and snow.
struct DayStatA {
  double m_prec, alpha, pet_mxdy, m_netrad, mcwh, t_snowfz, t_snowmt, t_gradnt;
  double melt_factor;          // M_DEGDAY_F * ddf_lct (daily.cpp:1013)
  double albedo, albedo_snow;
  double emis;                 // emissivity * 4.903e-9 (daily.cpp:423)
  double lmin, lmax;           // LAI limits (lai.cpp:78-89), float values
  int initial_days, lct, elev0;
  bool arid;                   // G_aindex == 1
};

// Statics of soil and local routing.
struct DayStatB {
  float built_up, smax, gw_factor;
  double gamma, cfa, pet_mxdy, t_snowfz, pcritgwa;
  double rgmax;                // G_Rgmax / 100
  bool recharge_cut;           // arid, texture < 21, no inland sink (daily.cpp:1166)
  bool arid;
  int ldd;
  double area, area_m;         // cell area, cell area / 1e6
  double cf100;                // contfreq / 100
  double fswb_catchment;       // min(1, 20 x initial surface-water fraction)
  double e_gw, inv_kgw, ome_gw, e_sw, k_sw;
  double red_exp;              // M_EVAREDEX * kEvapoRedExp
  double loc_lake, ll100, ll_max;        // percent, percent / 100, maximum storage
  double loc_wetland, lw100, lw_max;
  double glo_wetland, gw100, gw_max;
  double river_length, bottom, vel_b4, vel_b16, vel_c1, vel_c2;  // -B / 4, B B / 16
};

// Statics of global lakes and reservoirs, read for the cells that have one.
struct DayStatLake {
  double lake_area, lake_depth, reservoir_area, stor_cap, mean_outflow, prov_rel;
};

// Statics of the day's end.
struct DayStatEnd {
  double red_exp, area, river_length, rw_c0, rw_c1, rw_c2, rw_c3, river_stor_max;
  double max_raf;              // contfreq / 100 - f_glo_lake
  double f_glo_lake;
  double loc_lake, loc_wetland, glo_wetland, gw_max, lake_area, lake_max, reservoir_area, stor_cap;
  bool contcell;
};

// State that passes from day to day.
struct CellState {
  double canopy, soil, snow, transfer, lai_precsum;
  int lai_days, lai_status;
  bool snow_any;
  double gw, loc_lake, loc_wetl, glo_lake, glo_wetl, res, river;
  double red_ll, red_lw, red_gl, red_gw, red_res, red_river;
  double river_frac_next, river_frac_change, fswb_next, laf, laf_prev, k_release;
};

// Fluxes of the day passed between the parts.
struct DayFlux {
  double temp, prec, ow_pet, prec_to_soil, soil_pet, canopy_evapo, snow_evapo, eff_prec, temp_elev_max;
  double land_change, surf_runoff, recharge, aet;
};

// calcNewDay up to the canopy, daily.cpp:159-895 and lai.cpp:152-306: radiation,
// Priestley-Taylor PET, LAI, interception.  laf_prev: the fraction of daily.cpp:159-169.
__device__ __forceinline__ void day_pet_canopy(const DayStatA &a, CellState &s, DayFlux &v, float tf, float pf,
                                               float swf, float lwf, double laf_prev) {
  const double landAreaFrac = s.laf;
  double dailyTempC = tf, dailyPrec = pf;
  const double dailyShortWave = swf, dailyLongWave = lwf;
  dailyPrec = a.m_prec * dailyPrec;  // daily.cpp:248
  const double temp2 = dailyTempC + 237.3;
  const double e_s = 0.6108 * wg_exp(17.27 * dailyTempC / temp2);
  const double alpha = a.alpha;

  // lai.cpp:152-177
  const double dailyLai = lai_day(s.lai_days, a.initial_days, s.lai_status, a.lct, a.arid, a.lmin, a.lmax,
                                  s.lai_precsum, dailyPrec, dailyTempC > 8.);
  // daily.cpp:366-462 albedo, latent heat, radiation (cloud = 1)
  const double albedo = (s.snow > 3.) ? a.albedo_snow : a.albedo;
  const double lat_heat = (dailyTempC > 0) ? (2.501 - 0.002361 * dailyTempC) : 2.835;
  const double conv_Wm2_to_mmd = 0.0864 / lat_heat;
  const double solar_rad = conv_Wm2_to_mmd * dailyShortWave;
  const double long_wave_rad_in = conv_Wm2_to_mmd * dailyLongWave;
  const double temp_K = dailyTempC + 273.2;
  const double long_wave_rad_out = a.emis * wg_pow(temp_K, 4.) / lat_heat;
  const double net_long_wave_rad = long_wave_rad_in - long_wave_rad_out;
  const double net_short_wave_rad = solar_rad * (1. - albedo);
  const double net_rad = a.m_netrad * (net_short_wave_rad + net_long_wave_rad);
  const double openWaterNetRad = solar_rad * (1. - kOpenWaterAlbedo) + net_long_wave_rad;
  // daily.cpp:476-522 Priestley-Taylor
  const double inc_svp = 4098. * e_s / (temp2 * temp2);
  const double gamma = (0.0016286 * 101.3) / lat_heat;
  const double dailyPET = (net_rad <= 0.) ? 0. : alpha * (inc_svp * net_rad) / (inc_svp + gamma);
  const double dailyOpenWaterPET =
      (openWaterNetRad <= 0.) ? 0. : alpha * (inc_svp * openWaterNetRad) / (inc_svp + gamma);

  double dailyCanopyEvapo = 0., daily_prec_to_soil = 0., dailySoilPET = 0., change = 0.;
  // interception, daily.cpp:825-895
  double canopy = s.canopy;
  if (landAreaFrac <= 0.) {
    s.transfer = canopy;
    canopy = 0.;
  } else {
    canopy *= laf_prev / landAreaFrac;
    if (fabs(canopy) <= kMinStorVol) canopy = 0.;
    const double initialStorage = canopy;
    if (dailyLai > 0.00001) {
      const double max_canopy_storage = a.mcwh * dailyLai;
      const double canopy_deficiency = max_canopy_storage - canopy;
      if (dailyPrec < canopy_deficiency) {
        canopy += dailyPrec;
        daily_prec_to_soil = 0.;
      } else {
        canopy = max_canopy_storage;
        daily_prec_to_soil = dailyPrec - canopy_deficiency;
      }
      const double canopy_water_content = canopy;
      dailyCanopyEvapo = dailyPET * wg_pow((canopy_water_content / max_canopy_storage), kCanopyEvapoExp);
      if (dailyCanopyEvapo > canopy_water_content) {
        dailyCanopyEvapo = canopy_water_content;
        dailySoilPET = dailyPET - canopy_water_content;
        canopy = 0.0;
      } else {
        canopy -= dailyCanopyEvapo;
        dailySoilPET = dailyPET - dailyCanopyEvapo;
      }
    } else {
      daily_prec_to_soil = dailyPrec;
      dailySoilPET = dailyPET;
      dailyCanopyEvapo = 0.0;
    }
    change = 0. + (canopy - initialStorage);
  }
  s.canopy = canopy;
  if (dailySoilPET < 0.) dailySoilPET = 0.0;
  v.temp = dailyTempC;
  v.prec = dailyPrec;
  v.ow_pet = dailyOpenWaterPET;
  v.prec_to_soil = daily_prec_to_soil;
  v.soil_pet = dailySoilPET;
  v.canopy_evapo = dailyCanopyEvapo;
  v.land_change = change;
}

// Elevation extremes of a cell's sub-cells and its first sub-cell, for the test
// whether a whole day is bare.
struct ElevRange {
  int16_t lo, hi, first;
};

// One sub-cell of snow_subcell for finite storages 0 <= q (rescaled, before the
// zeroing of tiny ones), finite prec_to_soil and a melt factor > 0, with minima and
// maxima in place of most selects: precipitation pr and demand pe count only when
// freezing, so that max((s + pr) - pe, 0) is the storage after sublimation (s itself
// when not freezing) and min(pe, s + pr) the sublimation (0 then); the melt potential
// is negative or zero exactly when the temperature is not above M_T_SNOWMT, so its
// maximum with 0 is the melt demand and min(demand, s) the melt.  Each result is
// the reference's branch's, in value and rounding; a zero's sign may differ where
// it is only added to or subtracted from a sum that is not -0.
// kThresh: storages above 1,000 mm may occur (daily.cpp:958-976).
template <bool kThresh>
__device__ __forceinline__ double snow_subcell_fast(double q, double temp_elev, int elev_e, bool first,
                                                    const SnowDay &d, SnowAcc &a) {
  double s = (q <= kMinStorVol) ? 0. : q;
  const double init_s = s;
  if (kThresh) {
    const bool big = s > 1000.;
    const bool use_thresh = big && a.thresh > 0;
    const double temp_thresh = d.tempC - ((a.thresh - d.elev0) * d.gradnt);
    a.thresh = (big && a.thresh == 0) ? elev_e : a.thresh;
    temp_elev = use_thresh ? temp_thresh : temp_elev;
  }
  const bool freeze = temp_elev <= d.snowfz;
  const double pr = freeze ? d.prec_to_soil : 0.;
  const double pe = freeze ? d.soil_pet : 0.;
  const double s_fall = s + pr;
  a.evapo += fmin(pe, s_fall);
  s = fmax(s_fall - pe, 0.);
  const double demand = fmax(d.melt_factor * (temp_elev - d.snowmt), 0.);
  const double melt = fmin(demand, s);
  s = fmax(s - demand, 0.);
  a.change += s - init_s;
  if (first) a.temp_max = temp_elev;
  a.snow_sum += s;
  a.eff += (d.prec_to_soil - pr) + melt;
  return s;
}

// Snow on the elevation sub-cells of a cell with land (not s.laf <= 0), daily.cpp:897-1062,
// serial in sub-cell order.  Sub-cells are stored in pairs ([member][pair][cell] x 2 doubles, elevations as
// packed int16 pairs) and streamed in chunks, the next one loaded while one is
// stepped, so that a wavefront keeps many 16-byte loads in flight.  sub, elev: the member's pairs [k][n], cell p.
// What bounds it is a wavefront's instructions, issued and waited for one after the
// other: a sub-cell is 38 (61 before the minima and maxima of snow_subcell_fast), a bare
// one 2 additions' share; 100 of them are 25,300 of the 65,200 cycles of a day.
// kTwo: two load buffers, a chunk's loads out for the whole step of the chunk before
// (25 registers more); else one, refilled when its storages are rescaled.
template <int kSnowChunk, bool kTwo>
__device__ __forceinline__ void day_snow(const DayStatA &a, CellState &s, DayFlux &v, double laf_prev,
                                         const ElevRange &er, WgD2 *sub, const int32_t *elev, uint32_t p, int n) {
  auto sp = [&](int k) -> WgD2 & { return at(sub + int64_t(k) * n, p); };
  auto ep = [&](int k) -> int32_t { return at(elev + int64_t(k) * n, p); };
  SnowAcc acc;
  acc.snow_sum = 0.;
  acc.eff = 0.;
  acc.evapo = 0.;
  acc.change = 0.;
  acc.temp_max = 0.;
  acc.thresh = 0;
  // A cell whose sub-cell storages are all exactly zero (snow_any false) starts the
  // loop from zeros without reading them, and stores only storages that become
  // non-zero: on warm days such a cell moves no snow bytes at all.
  const bool snow_any = s.snow_any;
  SnowDay sd;
  sd.tempC = v.temp;
  sd.elev0 = a.elev0;
  sd.gradnt = a.t_gradnt;
  sd.scale_num = laf_prev;
  sd.laf = s.laf;
  sd.prec_to_soil = v.prec_to_soil;
  sd.soil_pet = v.soil_pet;
  sd.snowfz = a.t_snowfz;
  sd.snowmt = a.t_snowmt;
  sd.melt_factor = a.melt_factor;
  sd.inv_laf = 1. / s.laf;
  sd.melt_ok = sd.melt_factor > 0.;
  bool any_after = false;
  // The sub-cell temperature T - (z - z0) gradnt is monotonic in z, rounding
  // included, so the lowest and the highest sub-cell tell whether every sub-cell is
  // above freezing.  Without snow each of them then adds prec_to_soil + 0 to the
  // effective precipitation and nothing else: a wavefront of such cells reads no
  // sub-cell at all.  A land fraction that is not a number, of the day or the day
  // before, rescales no snow to NaN, which only the step of every sub-cell gives.
  const double t_lo = sd.tempC - ((er.lo - sd.elev0) * sd.gradnt);
  const double t_hi = sd.tempC - ((er.hi - sd.elev0) * sd.gradnt);
  const bool zero_stays = (0. * sd.scale_num) * sd.inv_laf == 0.;
  const bool bare_day = !snow_any && sd.melt_ok && t_lo > sd.snowfz && t_hi > sd.snowfz && zero_stays;
  if (__builtin_amdgcn_ballot_w64(!bare_day) == 0) {
    const double eff_bare = v.prec_to_soil + 0.;
    acc.temp_max = sd.tempC - ((er.first - sd.elev0) * sd.gradnt);
#pragma unroll 20
    for (int j = 0; j < 2 * WG_DEV_NPAIR; j++) acc.eff += eff_bare;
  } else {
    // snow_subcell_fast needs finite precipitation and a melt factor > 0.  (The test by
    // the high word keeps the instruction order that the step had without it: a year of
    // 6,485 cells with 8 members took 10.87 ms, and 10.95 with a comparison of doubles.)
    const bool usual = sd.melt_ok && (uint32_t(__double2hiint(sd.prec_to_soil)) & 0x7fffffffu) < 0x7ff00000u;
    WgD2 ia[kSnowChunk], ib[kSnowChunk];
    int32_t ea[kSnowChunk], eb[kSnowChunk];
    auto fetch = [&](int c, WgD2 *in, int32_t *en) {
#pragma unroll
      for (int j = 0; j < kSnowChunk; j++) {
        in[j] = snow_any ? sp(c * kSnowChunk + j) : WgD2{0., 0.};
        en[j] = ep(c * kSnowChunk + j);
      }
    };
    auto rescale = [&](const WgD2 *in, WgD2 *q) -> uint32_t {
      // The land-area rescaling s * scale_num / laf with the reused reciprocal:
      // q0 = x (1/laf), one exact residual and one correction give the correctly
      // rounded quotient (as in snow_subcell).  Storages in [0, 1000) mm, by the
      // high word of q, are the usual case; larger finite ones take the step with
      // the threshold elevation, anything else (negative, NaN, infinite, -0, or
      // not `usual`) the general step.
      uint32_t top = usual ? 0u : 0xffffffffu;
#pragma unroll
      for (int j = 0; j < kSnowChunk; j++) {
        const double x0 = in[j].x * sd.scale_num, y0 = in[j].y * sd.scale_num;
        const double rx = x0 * sd.inv_laf, ry = y0 * sd.inv_laf;
        q[j].x = fma(fma(-rx, sd.laf, x0), sd.inv_laf, rx);
        q[j].y = fma(fma(-ry, sd.laf, y0), sd.inv_laf, ry);
        top = max(top, max(uint32_t(__double2hiint(q[j].x)), uint32_t(__double2hiint(q[j].y))));
      }
      return top;
    };
    auto finish = [&](int c, WgD2 *q, const int32_t *en, uint32_t top) {
      if (__builtin_amdgcn_ballot_w64(top >= 0x7ff00000u) != 0) {
#pragma unroll 1
        for (int j = 0; j < kSnowChunk; j++) {
          const WgD2 w0 = snow_any ? sp(c * kSnowChunk + j) : WgD2{0., 0.};
          const int32_t ee = ep(c * kSnowChunk + j);
          const int e0 = int(int16_t(ee & 0xffff)), e1 = int(int16_t(ee >> 16));
          WgD2 w;
          w.x = snow_subcell(w0.x, sd.tempC - ((e0 - sd.elev0) * sd.gradnt), e0, c == 0 && j == 0, sd, acc);
          w.y = snow_subcell(w0.y, sd.tempC - ((e1 - sd.elev0) * sd.gradnt), e1, false, sd, acc);
          const bool nz = w.x != 0. || w.y != 0.;
          any_after |= nz;
          if (snow_any || nz) sp(c * kSnowChunk + j) = w;
        }
        return;
      }
      if (__builtin_amdgcn_ballot_w64(top >= 0x408f4000u) != 0) {
#pragma unroll
        for (int j = 0; j < kSnowChunk; j++) {
          const int e0 = int(int16_t(en[j] & 0xffff)), e1 = int(int16_t(en[j] >> 16));
          q[j].x = snow_subcell_fast<true>(q[j].x, sd.tempC - ((e0 - sd.elev0) * sd.gradnt), e0, c == 0 && j == 0, sd,
                                           acc);
          q[j].y = snow_subcell_fast<true>(q[j].y, sd.tempC - ((e1 - sd.elev0) * sd.gradnt), e1, false, sd, acc);
        }
      } else {
#pragma unroll
        for (int j = 0; j < kSnowChunk; j++) {
          const int e0 = int(int16_t(en[j] & 0xffff)), e1 = int(int16_t(en[j] >> 16));
          q[j].x = snow_subcell_fast<false>(q[j].x, sd.tempC - ((e0 - sd.elev0) * sd.gradnt), e0, c == 0 && j == 0,
                                            sd, acc);
          q[j].y = snow_subcell_fast<false>(q[j].y, sd.tempC - ((e1 - sd.elev0) * sd.gradnt), e1, false, sd, acc);
        }
      }
#pragma unroll
      for (int j = 0; j < kSnowChunk; j++) {
        const bool nz = q[j].x != 0. || q[j].y != 0.;
        any_after |= nz;
        if (snow_any || nz) sp(c * kSnowChunk + j) = q[j];
      }
    };
    constexpr int kChunks = WG_DEV_NPAIR / kSnowChunk;
    WgD2 q[kSnowChunk];
    fetch(0, ia, ea);
    if (kTwo) {
      static_assert(!kTwo || kChunks % 2 == 0, "chunks in pairs");
#pragma unroll 1
      for (int c = 0; c < kChunks; c += 2) {
        fetch(c + 1, ib, eb);
        finish(c, q, ea, rescale(ia, q));
        if (c + 2 < kChunks) fetch(c + 2, ia, ea);
        finish(c + 1, q, eb, rescale(ib, q));
      }
    } else {
#pragma unroll 1
      for (int c = 0; c < kChunks; c++) {
        const uint32_t top = rescale(ia, q);
#pragma unroll
        for (int j = 0; j < kSnowChunk; j++) eb[j] = ea[j];
        if (c + 1 < kChunks) fetch(c + 1, ia, ea);
        finish(c, q, eb, top);
      }
    }
  }
  s.snow_any = any_after;
  v.snow_evapo = acc.evapo / 100.;
  v.land_change += acc.change / 100.;
  v.temp_elev_max = acc.temp_max;
  v.eff_prec = acc.eff / 100.;
  s.snow = acc.snow_sum / 100.;
}

// The same for a cell without land: its snow leaves with the storage transfer.
__device__ __forceinline__ void day_snow_no_land(CellState &s, DayFlux &v, WgD2 *sub, uint32_t p, int n) {
  s.transfer += 0.;  // sub-cells without snow add 0
  if (s.snow_any) {
    for (int k = 0; k < WG_DEV_NPAIR; k++) {
      WgD2 &sp = at(sub + int64_t(k) * n, p);
      const WgD2 w = sp;
      s.transfer += w.x / 100.;
      s.transfer += w.y / 100.;
      sp = WgD2{0., 0.};
    }
  }
  s.snow_any = false;
  s.snow = 0.;
  v.snow_evapo = 0.;
  v.temp_elev_max = 0.;
  v.eff_prec = 0.;
}

// Immediate runoff, soil, runoff, AET and recharge, daily.cpp:1066-1257.
__device__ __forceinline__ void day_soil(const DayStatB &b, CellState &s, DayFlux &v, double laf_prev) {
  const double landAreaFrac = s.laf;
  double dailyEffPrec = v.eff_prec, immediate_runoff = 0., dailyAET = 0.;
  double daily_runoff = 0., total_daily_runoff = 0., daily_gw_recharge = 0., pot_gw_recharge = 0.;
  double soil_water_overflow = 0., neg_land_aet = 0., aet_uncorr = 0.;
  const float built_up = b.built_up;
  if (built_up > 0.) {
    immediate_runoff = kRunoffFracBuiltUp * dailyEffPrec * built_up;
    dailyEffPrec -= immediate_runoff;
  }
  // daily.cpp:1080-1239
  const double cfa = b.cfa;
  const float smax = b.smax;
  double soil = s.soil;
  if (landAreaFrac <= 0.) {
    s.transfer += soil;
    s.transfer *= cfa;
    soil = 0.;
    daily_gw_recharge = 0.;
    total_daily_runoff = 0.;
  } else {
    soil *= laf_prev / landAreaFrac;
    const double initialStorage = soil;
    soil_water_overflow = 0;
    if (soil > smax) {
      soil_water_overflow = soil - smax;
      soil = smax;
    }
    if (v.temp_elev_max > b.t_snowfz) {
      if (smax > 0.) {
        const double soil_saturation = soil / smax;
        daily_runoff = dailyEffPrec * wg_pow(soil_saturation, b.gamma);
        if (v.soil_pet > (b.pet_mxdy - v.canopy_evapo) * soil_saturation)
          dailyAET = (b.pet_mxdy - v.canopy_evapo) * soil_saturation;
        else
          dailyAET = v.soil_pet;
        soil += dailyEffPrec - dailyAET - daily_runoff;
        if (fabs(soil) <= kMinStorVol) soil = 0.;
        dailyEffPrec = 0.;
        if (soil < 0.) {
          dailyAET += soil;
          soil = 0.;
        }
        daily_runoff *= cfa;
        immediate_runoff *= cfa;
        const double rgmax = b.rgmax;
        const float fg = b.gw_factor;
        if (rgmax < (fg * daily_runoff))
          daily_gw_recharge = rgmax;
        else
          daily_gw_recharge = fg * daily_runoff;
        pot_gw_recharge = 0.;
        if (b.recharge_cut) {
          if (v.prec <= b.pcritgwa) {
            pot_gw_recharge = daily_gw_recharge;
            daily_gw_recharge = 0.;
          }
        }
        daily_runoff -= pot_gw_recharge;
        pot_gw_recharge /= cfa;
        soil += pot_gw_recharge;
        if (soil > smax) {
          soil_water_overflow += soil - smax;
          soil = smax;
        }
        soil_water_overflow *= cfa;
        total_daily_runoff = daily_runoff + immediate_runoff + soil_water_overflow;
      } else {
        total_daily_runoff = 0.;
        daily_gw_recharge = 0.;
      }
    } else {
      soil_water_overflow *= cfa;
      dailyEffPrec *= cfa;
      total_daily_runoff += soil_water_overflow + dailyEffPrec;
      daily_gw_recharge = 0.;
      dailyAET = 0.;
    }
    const double change = v.land_change + (soil - initialStorage);
    double cell_aet = change * (cfa - 1.0) - v.prec * (cfa - 1.0) +
                      (dailyAET + v.canopy_evapo + v.snow_evapo) * cfa;
    if (cell_aet < 0.) neg_land_aet = cell_aet;
    aet_uncorr = (dailyAET + v.canopy_evapo + v.snow_evapo);
  }
  // G_dailyGwRecharge is handed to routing before the corrections below (daily.cpp:1214)
  v.recharge = daily_gw_recharge;
  // surface runoff, daily.cpp:1241-1257
  if (neg_land_aet < 0.) total_daily_runoff = total_daily_runoff + neg_land_aet;
  if (total_daily_runoff < 0.) total_daily_runoff = 0.;
  if ((total_daily_runoff - daily_gw_recharge) < 0.) {
    const double neg_runoff = total_daily_runoff - daily_gw_recharge;
    daily_gw_recharge = total_daily_runoff;
    soil += neg_runoff;
  }
  v.surf_runoff = total_daily_runoff - daily_gw_recharge;
  v.aet = aet_uncorr;
  s.soil = soil;
}

// Terms of the potential cell runoff (optional output): the local runoff terms
// (routing.cpp:2045-2047 humid, 2180 inland sinks; (semi-)arid cells add their
// groundwater runoff with the routing step, 3372-3373) and the open-water
// precipitation minus evaporation of G_lakeBalance (daily.cpp:773).
struct PotTerms {
  double base, ow;
};

// Routing without upstream water, routing.cpp:1877-2617, and the routing record of
// the terms that do not depend on the inflow from upstream (2630-3514).  The
// chain constants and flags of c are set by the caller.  Updates the groundwater
// of humid cells and sinks, the local lake and the local wetland.
template <bool kUse>
__device__ __forceinline__ void day_local_routing(const DayStatB &b, const DayStatLake &lk, CellState &s,
                                                  const DayFlux &v, double use_desired, double use_nag, ChainRec &c,
                                                  PotTerms &pot) {
  const double cellArea = b.area;
  const int ldd = b.ldd;
  const double cfa = b.cfa;
  const double laf = s.laf;      // G_landAreaFrac of the day
  const double laf_prev = s.laf_prev;
  const double ow_prec = v.prec, ow_pet = v.ow_pet;
  double dailyLocalSurfaceRunoff, fswb_catchment = 0.;
  double localRunoff = 0., lrir = 0., lgwrir = 0., recharge_km3 = 0.;
  if (laf <= 0.)
    dailyLocalSurfaceRunoff = s.transfer * cellArea / 1000000. * laf_prev / 100.;
  else
    dailyLocalSurfaceRunoff = v.surf_runoff * cellArea / 1000000. * laf / 100.;
  if (ldd >= 0) {
    fswb_catchment = b.fswb_catchment;
    lrir = (1. - fswb_catchment) * dailyLocalSurfaceRunoff;
  }
  const bool arid_swb = b.arid && (ldd >= 0);
  const double gw_prev = s.gw;
  if (arid_swb) {
    localRunoff = fswb_catchment * dailyLocalSurfaceRunoff;
    recharge_km3 = v.recharge * cellArea * (laf / 100.) / 1000000.;
  } else {
    // humid cells (routing.cpp:1968-2039) and inland sinks (2112-2159)
    double netGWin = v.recharge * cellArea * (laf / 100.) / 1000000.;
    if (kUse) netGWin -= use_nag;  // routing.cpp:1990-1996, 2131-2137
    double gw = gw_prev * b.e_gw + b.inv_kgw * netGWin * b.ome_gw;
    if (fabs(gw) <= kMinStorVol) gw = 0.;
    double gw_runoff = gw_prev - gw + netGWin;
    if (gw_runoff <= 0.) {
      gw_runoff = 0.;
      gw = gw_prev + netGWin;
      if (fabs(gw) <= kMinStorVol) gw = 0.;
    }
    s.gw = gw;
    if (ldd >= 0) {
      lgwrir = (1. - fswb_catchment) * gw_runoff;
      const double localGWRunoff = fswb_catchment * gw_runoff;
      localRunoff = (fswb_catchment * dailyLocalSurfaceRunoff) + localGWRunoff;
    } else {
      if (laf == 0.)
        dailyLocalSurfaceRunoff = s.transfer * cellArea / 1000000. * laf_prev / 100.;
      else
        dailyLocalSurfaceRunoff = v.surf_runoff * cellArea / 1000000. * laf / 100.;
      localRunoff = dailyLocalSurfaceRunoff + gw_runoff;
    }
  }
  pot.base = (ldd < 0) ? localRunoff : (b.arid ? localRunoff + lrir : (localRunoff + lrir) + lgwrir);
  pot.ow = ow_prec - ow_pet;

  double inflow = localRunoff, outflow = 0.;
  double gwr_loclak = 0., gwr_locwet = 0.;
  // local lake, routing.cpp:2316-2490
  if (b.loc_lake > 0.) {
    const double prev = s.loc_lake, rf = s.red_ll;
    const double maxStorage = b.ll_max;
    double evap = ((1.0 - cfa) * ow_prec * rf) + (cfa * (ow_pet * rf));
    if (evap < 0.) evap = 0.;
    const double totalInflow = inflow + (ow_prec * rf) * b.area_m * b.ll100;
    if (arid_swb) gwr_loclak = kKswbgw * rf * b.loc_lake / 100. / b.cf100;
    const double PETgwr = evap * b.area_m * b.ll100 + gwr_loclak * cellArea * b.cf100 / 1000000.;
    double PETgwrMax = prev + maxStorage + totalInflow;
    if (PETgwrMax < 0.) PETgwrMax = 0.;
    double st;
    if (PETgwr > PETgwrMax) {
      st = (-1.) * maxStorage;
      gwr_loclak *= PETgwrMax / PETgwr;
    } else {
      st = prev + totalInflow - PETgwr;
    }
    if (prev > 0.) {
      outflow = b.k_sw * prev * wg_pow((prev / maxStorage), kLakeOutflowExp);
      if (st <= 0.) {
        outflow = 0;
      } else {
        if (outflow > st) outflow = st;
      }
    } else {
      outflow = 0.;
    }
    st -= outflow;
    if (fabs(st) <= kMinStorVol) st = 0.;
    if (st > maxStorage) {
      outflow += (st - maxStorage);
      st = maxStorage;
    }
    inflow = outflow;
    double r = 1. - wg_pow(fabs(st - maxStorage) / (2. * maxStorage), b.red_exp);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    s.loc_lake = st;
    s.red_ll = r;
  }
  // local wetland, routing.cpp:2495-2617
  if (b.loc_wetland > 0.) {
    const double prev = s.loc_wetl, rf = s.red_lw;
    const double maxStorage = b.lw_max;
    double evap = ((1.0 - cfa) * ow_prec * rf) + (cfa * (ow_pet * rf));
    if (evap < 0.) evap = 0.;
    const double totalInflow = inflow + (ow_prec * rf * b.area_m * b.lw100);
    if (arid_swb) gwr_locwet = kKswbgw * rf * b.loc_wetland / 100. / b.cf100;
    const double PETgwr = evap * b.area_m * b.lw100 + gwr_locwet * cellArea * b.cf100 / 1000000.;
    const double PETgwrMax = prev + totalInflow;
    double st;
    if (PETgwr > PETgwrMax) {
      st = 0.;
      gwr_locwet *= PETgwrMax / PETgwr;
    } else {
      st = prev + totalInflow - PETgwr;
    }
    if (fabs(st) <= kMinStorVol) st = 0.;
    if (st > 0.) {
      outflow = b.k_sw * st * wg_pow((st / maxStorage), kWetlOutflowExp);
      if (outflow > st) outflow = st;
    } else {
      outflow = 0.;
    }
    st -= outflow;
    if (st > maxStorage) {
      outflow += (st - maxStorage);
      st = maxStorage;
    }
    inflow = outflow;
    double r = 1. - wg_pow(fabs(st - maxStorage) / (maxStorage), b.red_exp);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    s.loc_wetl = st;
    s.red_lw = r;
  }

  double *w = c.v;
  const double e_sw = b.e_sw;
  {
    // river velocity and storage terms, routing.cpp:3424-3478
    const double L = b.river_length;
    const double prev = s.river;
    const double velocity = new_river_velocity(b.vel_c1, b.vel_c2, b.bottom, b.vel_b4, b.vel_b16, prev, L);
    const double K = velocity / L;
    const double eK = wg_exp(-1. * K);
    const double riverAreaFrac = s.river_frac_next;
    w[CF_INFLOW] = inflow;
    w[CF_LRIR] = lrir;
    w[CF_LGWRIR] = lgwrir;
    w[CF_RV_PREV] = prev;
    w[CF_RV_S0E] = prev * eK;
    w[CF_RV_INVK] = 1. / K;
    w[CF_RV_OME] = 1. - eK;
    w[CF_RV_TERM] = (K * prev * eK) / (1. - eK);
    w[CF_RV_EVAP] = ((1.0 - cfa) * (ow_prec) + (cfa * ow_pet)) * riverAreaFrac / 100. * cellArea / 1000000.;
    w[CF_RV_PREC] = ow_prec * riverAreaFrac / 100. * cellArea / 1000000.;
  }
  w[CF_OW_PREC] = ow_prec;
  w[CF_OW_PET] = ow_pet;
  {
    // global lake, routing.cpp:2633-2676
    w[CF_GL_LP] = 0.;
    w[CF_GL_USE] = 0.;
    w[CF_GL_MAX] = 0.;
    w[CF_GL_PREV] = 0.;
    w[CF_GL_S0E] = 0.;
    w[CF_GL_GWR] = 0.;
    const double lake_area = lk.lake_area;
    if (lake_area > 0.) {
      const double prev = s.glo_lake, rf = s.red_gl;
      double evap = ((1.0 - cfa) * ow_prec) + (cfa * ow_pet * rf);
      if (evap < 0.) evap = 0.;
      const double gwr = arid_swb ? kKswbgw * rf * (lake_area / (cellArea * b.cf100)) : 0.;
      w[CF_GL_MAX] = lake_area * lk.lake_depth;
      w[CF_GL_LP] = (ow_prec * (lake_area / 1000000.));
      w[CF_GL_GWR] = gwr;
      // the lake's share of the use, half of it when the cell has a reservoir too
      // (routing.cpp:2680-2695)
      const double use_lake = (c.flags & CFL_RES) ? 0.5 * use_desired : use_desired;
      w[CF_GL_USE] = evap * (lake_area / 1000000.) + gwr * cellArea * b.cf100 / 1000000. + (kUse ? use_lake : 0.);
      w[CF_GL_PREV] = prev;
      w[CF_GL_S0E] = prev * e_sw;
    }
  }
  {
    // global wetland, routing.cpp:3181-3222
    w[CF_GW_WP] = 0.;
    w[CF_GW_PET] = 0.;
    w[CF_GW_MAX] = 0.;
    w[CF_GW_PREV] = 0.;
    w[CF_GW_S0E] = 0.;
    w[CF_GW_GWR] = 0.;
    if (b.glo_wetland > 0) {
      const double prev = s.glo_wetl, rf = s.red_gw;
      double evap = ((1.0 - cfa) * (ow_prec * rf)) + (cfa * (ow_pet * rf));
      if (evap < 0.) evap = 0.;
      const double gwr = arid_swb ? kKswbgw * rf * b.glo_wetland / 100. / b.cf100 : 0.;
      w[CF_GW_MAX] = b.gw_max;
      w[CF_GW_WP] = (ow_prec * rf * b.area_m * b.gw100);
      w[CF_GW_GWR] = gwr;
      w[CF_GW_PET] = evap * b.area_m * b.gw100 + gwr * cellArea * b.cf100 / 1000000.;
      w[CF_GW_PREV] = prev;
      w[CF_GW_S0E] = prev * e_sw;
    }
  }
  {
    // groundwater of (semi-)arid cells, routing.cpp:3310-3330
    w[CF_A_GWR_LL] = gwr_loclak;
    w[CF_A_GWR_LW] = gwr_locwet;
    w[CF_A_RECH] = recharge_km3;
    const double gprev = arid_swb ? gw_prev : 0.;
    w[CF_A_PREV] = gprev;
    w[CF_A_S0E] = gprev * b.e_gw;
  }
  {
    // reservoir, routing.cpp:2807-2860 inputs
    const bool res = (c.flags & CFL_RES) != 0;
    w[CF_RES_PREV] = res ? s.res : 0.;
    w[CF_RES_RED] = res ? s.red_res : 0.;
    w[CF_RES_CFA] = cfa;
    w[CF_RES_KREL] = res ? s.k_release : 0.;
    w[CF_RES_CAP] = res ? lk.stor_cap : 0.;
    w[CF_RES_QMEAN] = res ? lk.mean_outflow : 0.;
    w[CF_RES_AREA] = res ? lk.reservoir_area : 0.;
    w[CF_RES_PROVREL] = res ? lk.prov_rel : 0.;
    w[CF_RES_PAD] = 0.;
  }
  w[CF_USE] = use_desired;
  w[CF_A_NUG] = use_nag;
}

// The use the river left, at the finished day's end (routing.cpp:3590-3622,
// 3898-3919): taken from the local lake, whose area reduction factor is recomputed;
// the unsatisfied use is kept and the month's irrigation withdrawal and
// consumptive use are recorded (fin_ym: model year x 12 + month of the finished
// day); after day 365 the year-end processing follows (fin_year_end).  U points at
// the member's first water-use field.
__device__ __forceinline__ void day_end_use(const WgStatic &S, double *U, uint32_t p, CellState &s, double rem,
                                            double loc_lake, double ll_max, double red_exp, int fin_ym,
                                            bool fin_year_end) {
  const int64_t us = S.use_stride;
  if ((loc_lake > 0.) && (rem > 0.)) {
    const double maxStorage = ll_max;
    double ls = s.loc_lake;
    if (ls > (-1.) * maxStorage) {
      if (rem < (maxStorage + ls)) {
        ls -= rem;
        rem = 0.;
      } else {
        rem -= (maxStorage + ls);
        ls = (-1.) * maxStorage;
      }
    }
    double r = 1. - wg_pow(fabs(ls - maxStorage) / (2. * maxStorage), red_exp);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    s.red_ll = r;
    s.loc_lake = ls;
  }
  if (S.use_delayed == 1) {
    const double tu = at(U + WG_USE_TOTAL_UNSAT * us, p);
    at(U + WG_USE_PREV_TOTAL_UNSAT * us, p) = tu;
    at(U + WG_USE_DAILY_REMAINING * us, p) = rem - tu;
    at(U + WG_USE_TOTAL_UNSAT * us, p) = rem;
  } else {
    at(U + WG_USE_TOTAL_UNSAT * us, p) += rem;
    at(U + WG_USE_DAILY_REMAINING * us, p) = rem;
  }
  const int64_t t = int64_t(fin_ym) * S.n;
  at(U + WG_USE_WITHDRAWAL_IRRIG * us, p) = at(S.use_wu + t, p);
  at(U + WG_USE_CONSUMPTIVE_IRRIG * us, p) = at(S.use_cu + t, p);
  if (fin_year_end) water_use_year_end(U, us, p);
}

// The end of a day: reduction factors of the global storages, river width and area
// fraction (routing.cpp:2792-2802, 3071-3078, 3286-3295, 3546-3586), then the
// surface-water and land area fractions (routing.cpp:5046-5174) and
// updateLandAreaFrac (routing.cpp:5343-5352).  s.red_gl and s.red_res change only
// in cells with such a storage.
__device__ __forceinline__ void day_end(const DayStatEnd &b, CellState &s) {
  const double cellArea = b.area;
  double red_ll = s.red_ll, red_lw = s.red_lw, red_gw = s.red_gw;
  double river_frac_next = s.river_frac_next, river_frac_change = s.river_frac_change, red_river = s.red_river;
  if (b.lake_area > 0.) {
    const double maxStorage = b.lake_max;
    double r = 1. - wg_pow(fabs(s.glo_lake - maxStorage) / (2. * maxStorage), b.red_exp);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    s.red_gl = r;
  }
  if (b.reservoir_area > 0.) {
    const double maxStorage = b.stor_cap;
    double r = 1. - wg_pow(fabs(s.res - maxStorage) / maxStorage, kEvapoRedExpRes);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    s.red_res = r;
  }
  if (b.glo_wetland > 0) {
    const double maxStorage = b.gw_max;
    double r = 1. - wg_pow(fabs(s.glo_wetl - maxStorage) / maxStorage, b.red_exp);
    if (r < 0.) r = 0.;
    if (r > 1.) r = 1.;
    red_gw = r;
  }
  if (b.contcell) {
    const double L = b.river_length, st = s.river, smax = b.river_stor_max;
    const double riverAreaFrac = river_frac_next;
    const double csa = st / L;
    // -B / (4. * 1000.), B / 1000. * B / (16. * 1000.), B / 1000. and width_bf / 1000.
    // are per-cell constants computed on the host with these operations
    const double depth = b.rw_c0 + sqrt(b.rw_c1 + 0.5 * csa);
    double width = b.rw_c2 + 4. * depth;
    if (width > b.rw_c3) width = b.rw_c3;
    red_river = 1. - wg_pow(fabs(st - smax) / smax, b.red_exp);
    if (red_river < 0.) red_river = 0.;
    if (red_river > 1.) red_river = 1.;
    river_frac_next = red_river * L * width * 100. / cellArea;
    river_frac_change = river_frac_next - riverAreaFrac;
  }
  // fractions for the next day
  const double loc_lake = b.loc_lake, loc_wetland = b.loc_wetland, glo_wetland = b.glo_wetland;
  double fLocLake, fLocWet, fGloWet;
  if ((loc_lake > 0.) && (red_ll > 0.))
    fLocLake = (red_ll * loc_lake / 100.);
  else
    fLocLake = 0.;
  if ((loc_wetland > 0.) && (red_lw > 0.))
    fLocWet = (red_lw * loc_wetland / 100.);
  else
    fLocWet = 0.;
  if ((glo_wetland > 0.) && (red_gw > 0.))
    fGloWet = (red_gw * glo_wetland / 100.);
  else
    fGloWet = 0.;
  double fswb_next = fLocLake + fLocWet + fGloWet;
  const double max_raf = b.max_raf;
  if (((b.lake_area > 0.) || (b.reservoir_area > 0.)) && (b.f_glo_lake == 1.)) {
    river_frac_next = 0.;
    river_frac_change = 0.;
    red_river = 0.;
  } else {
    if (river_frac_next <= max_raf) {
      if (fswb_next > (max_raf - river_frac_next)) {
        const double corr = (max_raf - river_frac_next) / fswb_next;
        red_ll *= corr;
        red_lw *= corr;
        red_gw *= corr;
        if ((fLocLake > 0.) && (red_ll > 0.)) {
          fLocLake = (red_ll * loc_lake / 100.);
        } else {
          red_ll = 0.;
          fLocLake = 0.;
        }
        if ((fLocWet > 0.) && (red_lw > 0.)) {
          fLocWet = (red_lw * loc_wetland / 100.);
        } else {
          red_lw = 0.;
          fLocWet = 0.;
        }
        if ((fGloWet > 0.) && (red_gw > 0.)) {
          fGloWet = (red_gw * glo_wetland / 100.);
        } else {
          red_gw = 0.;
          fGloWet = 0.;
        }
      }
    } else {
      const double deficit = river_frac_next - max_raf;
      river_frac_change -= deficit;
      red_river *= max_raf / river_frac_next;
      river_frac_next = max_raf;
      fLocLake = 0.;
      fLocWet = 0.;
      fGloWet = 0.;
    }
  }
  fswb_next = fLocLake + fLocWet + fGloWet;
  const double change_pct = fswb_next * 100. - s.fswb_next * 100.;
  const double laf = s.laf;
  double laf_next = laf - (change_pct + (river_frac_change * 100.));
  if (laf_next < 0.) laf_next = 0.;
  s.laf_prev = laf;
  s.laf = laf_next;
  s.fswb_next = fswb_next;
  s.red_ll = red_ll;
  s.red_lw = red_lw;
  s.red_gw = red_gw;
  s.red_river = red_river;
  s.river_frac_next = river_frac_next;
  s.river_frac_change = river_frac_change;
}

#endif  // WG_CELL_DAY_H
