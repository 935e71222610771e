"""The snow loop of a day (day_snow in watergap2_amd/csrc/wg_cell_day.h) takes one of
several steps per chunk of sub-cells: none on a bare day, one with minima and maxima
for storages below 1,000 mm, the same with the threshold elevation above, and the
general step (snow_subcell, daily.cpp:920-1044) for anything else.  Compiled for the
CPU with the kernels' floating-point flags, it must give the bits of a plain loop of
the general step over the 100 sub-cells, storages and sums, on random cells of every
kind: no snow, thin, tiny, deep and mixed storages, negative ones, -0, infinities and
NaN, odd parameters (melt temperature above or below freezing, zero, negative or NaN
factors, either sign of the gradient) and NaN precipitation or demand."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "watergap2_amd", "csrc")

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <type_traits>
#include <algorithm>
using std::fabs; using std::fma; using std::fmax; using std::fmin; using std::max; using std::min; using std::sqrt;
#define __device__
#define __forceinline__ inline
#include "../../include/watergap2_amd.h"
#include "wg_device.h"
#include "wg_libm.h"
#include "wg_route_step.h"
#define __builtin_amdgcn_ballot_w64(x) (uint64_t((x) ? 1 : 0))
static inline int __double2hiint(double v) { uint64_t b; std::memcpy(&b, &v, 8); return int(b >> 32); }
template <class T> T &at(T *row, uint32_t i) { return row[i]; }
#include "wg_cell_day.h"

static bool same(double a, double b) { return (a != a && b != b) || std::memcmp(&a, &b, 8) == 0; }

int main(int argc, char **argv) {
  const long n = std::atol(argv[1]);
  const bool unusual = argc > 2;
  std::mt19937_64 rng(11), odd_rng(12);
  std::uniform_real_distribution<double> U(0., 1.), W(0., 1.);
  const double inf = 1. / 0., nan = 0. / 0.;
  long bad = 0, bare = 0, deep = 0, odd = 0;
  for (long it = 0; it < n; it++) {
    DayStatA a{};
    CellState s{};
    DayFlux v{};
    const double kind = U(rng);
    a.t_snowfz = U(rng) < 0.7 ? 0. : 4. * U(rng) - 2.;
    a.t_snowmt = U(rng) < 0.7 ? 0. : 4. * U(rng) - 2.;
    a.t_gradnt = U(rng) < 0.85 ? 0.006 * U(rng) : (U(rng) < 0.5 ? -0.003 : 0.);
    a.melt_factor = U(rng) < 0.95 ? 8. * U(rng) : (U(rng) < 0.4 ? 0. : (U(rng) < 0.5 ? -1. : nan));
    WgD2 sub[50], ref[50];
    int32_t elev[50];
    const int base = int(U(rng) * 3000) - 100, spread = 1 + int(U(rng) * 4000);
    a.elev0 = base + int(U(rng) * spread);
    int lo = 1 << 20, hi = -(1 << 20), first = 0;
    for (int k = 0; k < 50; k++) {
      const int e0 = base + int(U(rng) * spread), e1 = base + int(U(rng) * spread);
      if (k == 0) first = e0;
      lo = min(lo, min(e0, e1));
      hi = max(hi, max(e0, e1));
      elev[k] = int32_t(uint32_t(uint16_t(int16_t(e0))) | uint32_t(uint16_t(int16_t(e1))) << 16);
    }
    auto one = [&]() -> double {
      if (kind < 0.25) return 0.;
      const double x = U(rng);
      if (kind < 0.5) return x < 0.2 ? 0. : (x < 0.3 ? 2e-15 * U(rng) : 300. * U(rng));
      if (kind < 0.7) return 990. + 20. * U(rng);
      if (kind < 0.9) return x < 0.5 ? 0. : 4000. * U(rng);
      return x < 0.8 ? 500. * U(rng) : (x < 0.85 ? -U(rng) : (x < 0.9 ? -0. : (x < 0.95 ? inf : nan)));
    };
    for (int k = 0; k < 50; k++) sub[k] = ref[k] = WgD2{one(), one()};
    s.snow_any = kind >= 0.25;
    s.laf = U(rng) < 0.1 ? 1e-14 * U(rng) + 1e-16 : 100. * U(rng) + 1e-3;
    double laf_prev = U(rng) < 0.5 ? s.laf : 100. * U(rng);
    v.temp = float(30. * U(rng) - 15.);
    v.prec_to_soil = U(rng) < 0.3 ? 0. : 20. * U(rng);
    v.soil_pet = U(rng) < 0.3 ? 0. : 6. * U(rng);
    if (U(rng) < 0.01) v.prec_to_soil = nan;
    if (U(rng) < 0.01) v.soil_pet = nan;
    if (unusual) {  // land fractions that are no positive numbers (a state from NaN storages)
      const double x = W(odd_rng);
      if (x < 0.3) s.laf = nan;
      if (x > 0.2 && x < 0.5) laf_prev = x < 0.35 ? nan : inf;
      // and weather and parameters that overflowed (a perturbation's exponential)
      auto some = [&](double &y, double z) { if (W(odd_rng) < 0.1) y = z; };
      some(v.prec_to_soil, inf);
      some(v.prec_to_soil, -inf);
      some(v.soil_pet, inf);
      some(v.temp, W(odd_rng) < 0.6 ? inf : (W(odd_rng) < 0.5 ? -inf : nan));
      some(a.melt_factor, W(odd_rng) < 0.5 ? inf : 0.);
      some(a.t_snowmt, W(odd_rng) < 0.5 ? inf : -inf);
      some(a.t_snowfz, W(odd_rng) < 0.5 ? inf : -inf);
      some(a.t_gradnt, W(odd_rng) < 0.5 ? inf : 1e306);
    }
    // the general step over all sub-cells
    SnowDay sd{};
    sd.tempC = v.temp; sd.gradnt = a.t_gradnt; sd.scale_num = laf_prev; sd.laf = s.laf;
    sd.prec_to_soil = v.prec_to_soil; sd.soil_pet = v.soil_pet; sd.snowfz = a.t_snowfz; sd.snowmt = a.t_snowmt;
    sd.melt_factor = a.melt_factor; sd.inv_laf = 1. / s.laf; sd.elev0 = a.elev0;
    SnowAcc acc{};
    bool any = false;
    for (int k = 0; k < 50; k++) {
      const int e0 = int16_t(elev[k] & 0xffff), e1 = int16_t(elev[k] >> 16);
      ref[k].x = snow_subcell(ref[k].x, sd.tempC - ((e0 - sd.elev0) * sd.gradnt), e0, k == 0, sd, acc);
      ref[k].y = snow_subcell(ref[k].y, sd.tempC - ((e1 - sd.elev0) * sd.gradnt), e1, false, sd, acc);
      any |= ref[k].x != 0. || ref[k].y != 0.;
    }
    bare += !s.snow_any && !any;
    deep += acc.thresh != 0;
    odd += kind >= 0.9;
    const ElevRange er{int16_t(lo), int16_t(hi), int16_t(first)};
    if (it % 3 == 0) day_snow<5, true>(a, s, v, laf_prev, er, sub, elev, 0, 1);
    else if (it % 3 == 1) day_snow<5, false>(a, s, v, laf_prev, er, sub, elev, 0, 1);
    else day_snow<10, false>(a, s, v, laf_prev, er, sub, elev, 0, 1);
    bool ok = same(s.snow, acc.snow_sum / 100.) && same(v.eff_prec, acc.eff / 100.) &&
              same(v.snow_evapo, acc.evapo / 100.) && same(v.land_change, 0. + acc.change / 100.) &&
              same(v.temp_elev_max, acc.temp_max) && s.snow_any == any;
    for (int k = 0; k < 50; k++) ok = ok && same(sub[k].x, ref[k].x) && same(sub[k].y, ref[k].y);
    if (!ok && bad++ < 5) std::printf("mismatch %ld kind %.2f laf %g T %g\n", it, kind, s.laf, v.temp);
  }
  std::printf("%ld %ld %ld %ld %ld\n", n, bad, bare, deep, odd);
  return 0;
}
"""


def snow_loop(tmp_path, *args):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    src, exe = str(tmp_path / "snow.cpp"), str(tmp_path / "snow")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-w", "-I", CSRC, src, "-o", exe],
                   check=True)
    out = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout
    n, bad, bare, deep, odd = map(int, out.strip().splitlines()[-1].split())
    assert bad == 0, out
    return n, bare, deep, odd


def test_snow_loop_gives_the_general_steps_bits(tmp_path):
    n, bare, deep, odd = snow_loop(tmp_path, "60000")
    assert bare > n // 20 and deep > n // 10 and odd > n // 20


def test_snow_loop_of_unusual_cells(tmp_path):
    """Land fractions that are no positive numbers, infinite or huge weather and
    parameters: the step that a cell takes does not depend on its neighbours in the
    wavefront, nor on the days of a call."""
    snow_loop(tmp_path, "60000", "unusual")
