// cbm_step.h -- the per-tile CABLE timestep on the GPU (device code).
//
// Stepper<R, FULL, TABLES, MODE, V>::run() performs, for the tile held in `t`,
// one call of the reference's cbm() together with the offline driver's
// contract around it; see cbm_physics.h for the template parameters and
// layout.  MODE (StepMode) adds the surrogate's work: MODE_CAPTURE records
// the converged leaf state as a training target; MODE_HYBRID starts the leaf
// fixed point from the surrogate's prediction, caps its passes and reports
// whether the tile must fall back to the plain method; MODE_UNLIT is the plain
// method that also keeps the leaf state the next step's surrogate inputs read.
#pragma once
#include "cbm_physics.h"

namespace cbm {

template <class R, bool FULL, bool TABLES, int MODE = MODE_PLAIN, class V = double, bool DERIVED = false>
struct Stepper {
  Tile<R> &t;
  const StepArgs &a;
  const ClassRows<V> rows;
  int npass = 0;
  // surrogate: predictions in (MODE_HYBRID), targets out (MODE_CAPTURE), and
  // whether a capped tile's leaf fixed point fell back to the reference's
  // iteration (MODE_HYBRID)
  float pred[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float tgt[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  bool fell_back = false;
  bool vegetated = false;
  bool capped = false;         // MODE_HYBRID: a sunlit leaf-bearing tile, whose
                               // leaf passes are capped and checked
  float *hyb_out = nullptr;     // MODE != MODE_PLAIN: the tile's leaf temperature,
                               // canopy-air temperature and humidity, `a.mp` apart

  // ---- constants: src/params/*, src/util/cable_common.F90:217-222 ----
  static constexpr R TFRZ = R(273.16), SBOLTZ = R(5.67e-8), EMSOIL = R(1.0),
                     EMLEAF = R(1.0), CAPP = R(1004.64), HL = R(2.5014e6),
                     HLF = R(0.334e6), DHEAT = R(21.5e-6), GRAV = R(9.8086),
                     RGAS = R(8.3143), RMAIR = R(0.02897), RMH2O = R(0.018016),
                     CGSNOW = R(2090.0), CSICE = R(2.100e3), CSWAT = R(4.218e3),
                     DENSITY_LIQ = R(1000.0), DENSITY_ICE = R(921.0),
                     TETENA = R(6.106), TETENB = R(17.27), TETENC = R(237.3),
                     VONK = R(0.40), A33 = R(1.25), CSW = R(0.50), CTL = R(0.40),
                     APOL = R(0.70), PRANDT = R(0.71), CRD = R(0.3), CSD = R(0.003),
                     CCD = R(15.0), CCW_C = R(2.0), USUHM = R(0.3), ZETA0 = R(0.0),
                     ZETNEG = R(-15.0), ZETPOS = R(1.0), ZDLIN = R(1.0), UMIN = R(0.1),
                     PI_C = R(3.1415927), LAI_THRESH = R(0.001), RAD_THRESH = R(0.001),
                     COSZEN_TOLS = R(1.0e-4), GAM0 = R(28.0e-6), GAM1 = R(0.0509),
                     GAM2 = R(0.0010), RGBWC = R(1.32), RGSWC = R(1.57),
                     TREFK = R(298.2), MAX_GLACIER_SNOWD = R(1100.0),
                     SNOW_CCNSW = R(2.0), MAX_SSDN = R(750.0), MAX_SCONDS = R(2.51),
                     FROZEN_LIMIT = R(0.85), SNMIN = R(1.0);
  static constexpr int LAKES = 16, ICE_VEG = 17, ICE_SOIL = 9;

  CBM_HD Stepper(Tile<R> &t_, const StepArgs &a_, const ClassRows<V> &r) : t(t_), a(a_), rows(r) {}

  // a / b and x**0.5.  The plain path takes them on the device as the short
  // sequences of cbm_physics.h: the same bits as the compiler's IEEE
  // sequences at four fifths of the instructions.  Written out, a
  // reciprocal is shared by the quotients of one divisor and leaves the leaf
  // iteration where the divisor is fixed, and a constant's is folded.
  // Divisions were a third of the FP64 step's instructions.  Static VALU
  // instructions of the resident FP64 step 17,561 -> 14,980; a step of 4,093
  // tiles 146 -> 129 us, of 262,144 tiles 445 -> 421 us (day average, with
  // the read-back)
  template <class A, class B>
  CBM_HD static auto DIV(A a, B b) -> decltype(a / b) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(R) == 8) {
      const double r = __builtin_constant_p(b) ? 1.0 / b : refine_reciprocal(b, __builtin_amdgcn_rcp((double)b));
      return __builtin_amdgcn_div_fixup(corrected_quotient(a, b, r), (double)b, (double)a);
    }
#endif
    return a / b;
  }
  // DIV(a, b) with r = recip(b)
  CBM_HD static R recip(R b) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(R) == 8) return refine_reciprocal(b, __builtin_amdgcn_rcp((double)b));
    else return __builtin_amdgcn_rcpf((float)b);
#else
    return K(1.0) / b;
#endif
  }
  CBM_HD static R DIVR(R a, R b, R r) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(R) == 8)
      return __builtin_amdgcn_div_fixup(corrected_quotient(a, b, r), (double)b, (double)a);
    else
      return a * r;
#else
    return a / b;
#endif
  }
  // a derived column (ClassRows::x) from its vegetation row
  template <class P>
  CBM_HD static R derived(int c, P &&veg) {
    switch (c) {
      case VX_rdleaf: return recip(veg(VC_dleaf));
      case VX_dleaf3: return p3(veg(VC_dleaf));
      case VX_r2convex: return recip(K(2.0) * veg(VC_convex));
      case VX_c4ca: return K(4.0) * veg(VC_convex) * veg(VC_alpha);
      case VX_rd0gs: return recip(veg(VC_d0gs));
      case VX_ekc: return DIV(veg(VC_ekc), RGAS * TREFK);
      default: return DIV(veg(VC_eko), RGAS * TREFK);
    }
  }
  CBM_HD R derived(int c) const {
    if constexpr (DERIVED) {
      return rows.x[c];
    } else {
      return derived(c, [&](int v) {
        return v == VC_dleaf    ? PV(veg_dleaf, 0)
               : v == VC_convex ? PV(veg_convex, 0)
               : v == VC_alpha  ? PV(veg_alpha, 0)
               : v == VC_d0gs   ? PV(veg_d0gs, 0)
               : v == VC_ekc    ? PV(veg_ekc, 0)
                                : PV(veg_eko, 0);
      });
    }
  }
  template <class T>
  CBM_HD static T sqrt(T x) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(R) == 8 && sizeof(T) == 8) {
      const T g = refined_root(x, __builtin_amdgcn_rsq(x));
      return x == 0.0 || x == __builtin_inf() ? x : g;
    }
#endif
    return std::sqrt(x);
  }
  // x**0.25 and x**1.5 for x >= 0 through the square root: within about an
  // ulp of pow (two correctly rounded steps), at a small part of the cost of
  // the FP64 pow sequence
  CBM_HD static R root4(R x) { return sqrt(sqrt(x)); }
  CBM_HD static R pow1p5(R x) { return x * sqrt(x); }

  // ===================================================================
  // src/science/roughness/roughnessHGT_effLAI_cbl.F90:42-149,
  // src/science/roughness/cable_roughness.F90:64-317
  CBM_HD void ruff_resist() {
    const R z0soilsn_min = K(1.e-7), z0soilsn_min_PF = K(1.e-4);
    R sde = MAX(K(100.0), t.ssnow_ssdnn[0]);
    R hmin = K(10.0) * z0soilsn_min;
    R hc = PV(veg_hc, 0);
    R hcomp = hc - DIV(K(1.2) * t.ssnow_snowd[0], sde);
    R hruff = MAX(hmin, hcomp);
    t.rough_hruff[0] = hruff;
    R frac = DIV(hruff, MAX(K(0.01), hc));
    R vlaiw = t.veg_vlai[0] * frac;
    t.canopy_vlaiw[0] = vlaiw;
    t.canopy_rghlai[0] = vlaiw;
    R z0soil = K(0.0009) * MIN(K(1.0), vlaiw) + K(1.e-4);
    R z0soilsn = z0soil;
    R snowd = t.ssnow_snowd[0];
    if (snowd > K(0.01))
      z0soilsn = MAX(z0soilsn_min, z0soil - DIV(z0soil * MIN(snowd, K(10.)), K(10.)));
    if (snowd > K(0.01) && t.veg_iveg[0] == ICE_VEG) z0soilsn = MAX(z0soilsn, z0soilsn_min_PF);
    t.rough_z0soil[0] = z0soil;
    t.rough_z0soilsn[0] = z0soilsn;
    R rghlai = vlaiw;
    R za_uv = PV(rough_za_uv, 0), za_tq = PV(rough_za_tq, 0);
    if (vlaiw <= LAI_THRESH || hruff < z0soilsn) {
      R z0m = z0soilsn;
      t.rough_z0m[0] = z0m;
      t.rough_rt0us[0] = K(0.0);
      t.rough_disp[0] = K(0.0);
      R zuv = MAX(K(3.5) + z0m, za_uv);
      R ztq = MAX(K(3.5) + z0m, za_tq);
      zuv = MAX(zuv, hruff - K(0.0));
      ztq = MAX(ztq, hruff - K(0.0));
      t.rough_zref_uv[0] = zuv;
      t.rough_zref_tq[0] = ztq;
      t.rough_zruffs[0] = K(0.0);
      t.rough_rt1usa[0] = K(0.0);
      t.rough_rt1usb[0] = K(0.0);
      R usuh = MIN(sqrt(CSD + CRD * (vlaiw * K(0.5))), USUHM);
      R xx = sqrt(CCD * MAX((vlaiw * K(0.5)), K(0.0005)));
      R dh = K(1.0) - DIV(K(1.0) - exp(-xx), xx);
      t.rough_usuh[0] = usuh;
      t.rough_coexp[0] = DIV(usuh, VONK * CCW_C * (K(1.0) - dh));
    } else {
      R usuh = MIN(sqrt(CSD + CRD * (rghlai * K(0.5))), USUHM);
      R xx = sqrt(CCD * MAX((rghlai * K(0.5)), K(0.0005)));
      R dh = K(1.0) - DIV(K(1.0) - exp(-xx), xx);
      R disp = dh * hruff;
      R z0m = ((K(1.0) - dh) * exp(log(CCW_C) - K(1.) + K(1.) / CCW_C - DIV(VONK, usuh))) * hruff;
      R zuv = MAX(K(3.5) + z0m, za_uv);
      R ztq = MAX(K(3.5) + z0m, za_tq);
      zuv = MAX(zuv, hruff - disp);
      ztq = MAX(ztq, hruff - disp);
      R coexp = DIV(usuh, VONK * CCW_C * (K(1.0) - dh));
      R term2 = exp(K(2) * CSW * rghlai * (K(1) - DIV(disp, hruff)));
      R term3 = A33 * A33 * CTL * K(2) * CSW * rghlai;
      R term5 = MAX(DIV((K(2.) / K(3.)) * hruff, disp), K(1.0));
      R term6 = exp(K(3.) * coexp * (DIV(disp, hruff) - K(1.)));
      R term6a = exp(coexp * (DIV(K(0.1) * hruff, hruff) - K(1.)));
      R rt0us = DIV(term5 * (ZDLIN * log(DIV(ZDLIN * disp, z0soilsn)) + (K(1) - ZDLIN)) *
                (exp(K(2) * CSW * rghlai) - term2), term3);
      R zruffs = disp + DIV(DIV(hruff * (A33 * A33) * CTL, VONK), term5);
      R rt1usa = DIV(term5 * (term2 - K(1.0)), term3);
      R rt1usb = DIV(term5 * (MIN(ztq + disp, zruffs) - hruff), A33 * A33 * CTL * hruff);
      rt1usb = MAX(rt1usb, K(0.0));
      t.rough_usuh[0] = usuh;
      t.rough_disp[0] = disp;
      t.rough_z0m[0] = z0m;
      t.rough_zref_uv[0] = zuv;
      t.rough_zref_tq[0] = ztq;
      t.rough_coexp[0] = coexp;
      t.rough_term2[0] = term2;
      t.rough_term3[0] = term3;
      t.rough_term5[0] = term5;
      t.rough_term6[0] = term6;
      t.rough_term6a[0] = term6a;
      t.rough_rt0us[0] = rt0us;
      t.rough_zruffs[0] = zruffs;
      t.rough_rt1usa[0] = rt1usa;
      t.rough_rt1usb[0] = rt1usb;
    }
  }

  // src/science/misc/cable_air.F90:51-97
  CBM_HD void define_air() {
    R tv = t.met_tvair[0], pmb = t.met_pmb[0];
    R es = TETENA * exp(DIV(TETENB * (tv - TFRZ), TETENC + (tv - TFRZ)));
    R cmolar = DIV(pmb * K(100.0), RGAS * (tv));
    t.air_cmolar[0] = cmolar;
    t.air_rho[0] = MIN(K(1.3), RMAIR * cmolar);
    t.air_volm[0] = DIV(RGAS * (tv), K(100.0) * pmb);
    R rlam = HL;
    t.air_rlam[0] = rlam;
    t.air_qsat[0] = DIV((RMH2O / RMAIR) * es, pmb);
    t.air_epsi[0] = DIV(DIV(DIV(rlam, CAPP) * (RMH2O / RMAIR) * es * TETENB * TETENC,
                    p2(TETENC + (tv - TFRZ))), pmb);
    t.air_visc[0] = K(1e-5) * MAX(K(1.0), K(1.35) + K(0.0092) * (tv - TFRZ));
    t.air_psyc[0] = DIV(DIV(pmb * K(100.0) * CAPP * RMAIR, rlam), RMH2O);
    t.air_dsatdk[0] = DIV(K(100.0) * (TETENA * TETENB * TETENC), p2((tv - TFRZ) + TETENC)) *
                      exp(DIV(TETENB * (tv - TFRZ), (tv - TFRZ) + TETENC));
  }

  // src/science/canopy/cbl_qsat.F90:16-53
  CBM_HD static R qsatfjh(R tair, R pmb) {
    return DIV((RMH2O / RMAIR) * (TETENA * exp(DIV(TETENB * tair, TETENC + tair))), pmb);
  }

  // src/science/radiation/cbl_spitter.F90:36-76
  CBM_HD static R spitter(int doy, R coszen, R fsd) {
    const R solcon = K(1370.0);
    R fbeam = K(0.0), tmprat;
    R tmpr = K(0.847) + coszen * (K(1.04) * coszen - K(1.61));
    R tmpk = DIV(K(1.47) - tmpr, K(1.66));
    if (coszen > K(1.0e-10) && fsd > K(10.0))
      tmprat = DIV(fsd, solcon * (K(1.0) + K(0.033) * cos(DIV(K(2.0) * PI_C * ((R)doy - K(10.0)),
                                                        K(365.0)))) * coszen);
    else
      tmprat = K(0.0);
    if (tmprat > K(0.22)) fbeam = K(6.4) * p2(tmprat - K(0.22));
    if (tmprat > K(0.35)) fbeam = MIN(K(1.66) * tmprat - K(0.4728), K(1.0));
    if (tmprat > tmpk) fbeam = MAX(K(1.0) - tmpr, K(0.0));
    return fbeam;
  }

  // src/science/radiation/cbl_init_radiation.F90:30-392, cbl_rhoch.F90:38-62,
  // src/science/albedo/cbl_albedo.F90:56-386, cbl_snow_albedo.F90:36-161
  CBM_HD void init_radiation_albedo(bool veg_mask) {
    const R pi180 = PI_C / K(180.0);
    const R GW0 = K(0.308), GW1 = K(0.514), GW2 = K(0.178);
    R vlaiw = t.canopy_vlaiw[0], coszen = t.met_coszen[0];
    R cos3[3] = {cos(pi180 * K(15.0)), cos(pi180 * K(45.0)), cos(pi180 * K(75.0))};
    R xphi1 = K(0.0), xphi2 = K(0.0);
    if (veg_mask) {
      R xf = PV(veg_xfang, 0);
      xphi1 = K(0.5) - xf * (K(0.633) + K(0.33) * xf);
      xphi2 = K(0.877) * (K(1.0) - K(2.0) * xphi1);
    }
    R xk[3], c1[3], rhoch[3];
#pragma unroll
    for (int b = 0; b < 3; b++) xk[b] = (vlaiw > LAI_THRESH) ? DIV(xphi1, cos3[b]) + xphi2 : K(0.0);
    c1[0] = sqrt(K(1.0) - PV(veg_taul, 0) - PV(veg_refl, 0));
    c1[1] = sqrt(K(1.0) - PV(veg_taul, 1) - PV(veg_refl, 1));
    c1[2] = K(1.0);
#pragma unroll
    for (int b = 0; b < 3; b++) rhoch[b] = DIV(K(1.0) - c1[b], K(1.0) + c1[b]);
    R tiny = COSZEN_TOLS * K(1e-2), huge = COSZEN_TOLS * K(1e2);
    R extkb = K(0.5), extkd = K(0.7);
    if (veg_mask) {
      R s = GW0 * exp(-xk[0] * vlaiw);
      s = s + GW1 * exp(-xk[1] * vlaiw);
      s = s + GW2 * exp(-xk[2] * vlaiw);
      extkd = DIV(-log(s), vlaiw);
    }
    if (veg_mask && coszen > tiny) extkb = DIV(xphi1, coszen) + xphi2;
    if (coszen < tiny) extkb = K(1.0e5);
    if (fabs(extkb - extkd) < K(0.001)) extkb = extkd + K(0.001);
    t.rad_extkb[0] = extkb;
    t.rad_extkd[0] = extkd;
#pragma unroll
    for (int b = 0; b < 3; b++) t.rad_extkbm[b] = K(0.0), t.rad_extkdm[b] = K(0.0);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (veg_mask) t.rad_extkbm[b] = extkb * c1[b];
      t.rad_extkdm[b] = extkd * c1[b];
    }
    R fb = spitter((int)t.met_doy[0], coszen, t.met_fsd[0] + t.met_fsd[1]);
    t.rad_fbeam[0] = fb;
    t.rad_fbeam[1] = fb;
    if (coszen < huge) t.rad_fbeam[0] = K(0.0), t.rad_fbeam[1] = K(0.0);

    // Albedo
    R alb[3] = {K(0.0), K(0.0), K(0.0)};
#pragma unroll
    for (int b = 0; b < 3; b++) t.rad_rhocbm[b] = K(0.0), t.rad_rhocdf[b] = K(0.0);
    {
      const R alvo = K(0.95), aliro = K(0.70);
      int iveg = t.veg_iveg[0];
      R snowd = t.ssnow_snowd[0];
      R sa = t.soil_albsoil[0];
      if (iveg == LAKES)
        sa = -K(0.022) * (MIN(K(275.0), MAX(K(260.0), t.ssnow_tgg[0])) - K(260.0)) + K(0.45);
      if (snowd > K(1.0) && iveg == LAKES) sa = K(0.85);
      R sfact = K(0.68);
      if (sa <= K(0.14))
        sfact = K(0.5);
      else if (sa > K(0.14) && sa <= K(0.20))
        sfact = K(0.62);
      alb[1] = DIV(K(2.0) * sa, K(1.0) + sfact);
      alb[0] = sfact * alb[1];
      R snrat = K(0.0), alir = K(0.0), alv = K(0.0);
      if (snowd > K(1.0)) {
        R tmp = DIV(snowd, MAX(t.ssnow_ssdnn[0], K(200.0)));
        snrat = MIN(K(1.0), DIV(tmp, tmp + K(0.1)));
        R fage = K(1.0) - DIV(K(1.0), K(1.0) + t.ssnow_snage[0]);
        tmp = MAX(K(0.17365), coszen);
        R fz = (tmp > K(0.5)) ? K(0.0) : DIV(K(1.5), K(1.0) + K(4.0) * tmp) - K(0.5);
        R fzenm = MAX(K(0.0), fz);
        tmp = alvo * (K(1.0) - K(0.2) * fage);
        alv = K(0.4) * fzenm * (K(1.0) - tmp) + tmp;
        tmp = aliro * (K(1.0) - K(0.5) * fage);
        alir = K(0.4) * fzenm * (K(1.0) - tmp) + tmp;
      }
      alb[1] = MIN(aliro, (K(1.0) - snrat) * alb[1] + snrat * alir);
      alb[0] = MIN(alvo, (K(1.0) - snrat) * alb[0] + snrat * alv);
      if (t.soil_isoilm[0] == ICE_SOIL) {
        alb[0] = alvo - K(0.05);
        alb[1] = aliro - K(0.05);
      }
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (veg_mask) t.rad_rhocbm[b] = DIV(K(2.0) * extkb, extkb + extkd) * rhoch[b];
      t.rad_rhocdf[b] = rhoch[b] * K(2.0) *
                        (DIV(GW0 * xk[0], xk[0] + extkd) + DIV(GW1 * xk[1], xk[1] + extkd) +
                         DIV(GW2 * xk[2], xk[2] + extkd));
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (veg_mask) {
        R d = MIN(t.rad_extkbm[b] * vlaiw, K(20.0));
        t.rad_cexpkbm[b] = exp(-K(1.0) * d);
      }
      R d = t.rad_extkdm[b] * vlaiw;
      t.rad_cexpkdm[b] = exp(-K(1.0) * d);
    }
#pragma unroll
    for (int b = 0; b < 3; b++) t.rad_reffbm[b] = alb[b], t.rad_reffdf[b] = alb[b];
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (veg_mask) {
        t.rad_reffdf[b] = t.rad_rhocdf[b] + (alb[b] - t.rad_rhocdf[b]) * p2(t.rad_cexpkdm[b]);
        t.rad_reffbm[b] = t.rad_rhocbm[b] + (alb[b] - t.rad_rhocbm[b]) * p2(t.rad_cexpkbm[b]);
      }
    }
#pragma unroll
    for (int b = 0; b < 3; b++) t.rad_albedo[b] = alb[b];
#pragma unroll
    for (int b = 0; b < 2; b++)
      if (veg_mask)
        t.rad_albedo[b] = (K(1.0) - t.rad_fbeam[b]) * t.rad_reffdf[b] + t.rad_fbeam[b] * t.rad_reffbm[b];
#pragma unroll
    for (int b = 0; b < 3; b++) t.ssnow_albsoilsn[b] = alb[b];
  }

  // src/science/radiation/cbl_radiation.F90:30-218
  CBM_HD void radiation(bool sunlit_veg) {
    R vlaiw = t.canopy_vlaiw[0];
    R extkb = t.rad_extkb[0], extkd = t.rad_extkd[0];
    R extkn = PV(veg_extkn, 0);
    R cf2n = exp(-extkn * vlaiw);
    R transd = K(1.0);
    if (vlaiw > LAI_THRESH) transd = exp(-extkd * vlaiw);
    R dummy2 = MIN(extkb * vlaiw, K(30.));
    R transb = exp(-dummy2);
    t.rad_transd[0] = transd;
    t.rad_transb[0] = transb;
    R tvrad = t.met_tvrad[0];
    R flpwb = SBOLTZ * p4(tvrad);
    R flwv = EMLEAF * flpwb;
    R flws = SBOLTZ * EMSOIL * p4(t.ssnow_tss[0]);
    t.rad_flws[0] = flws;
    R emair = DIV(t.met_fld[0], flpwb);
    R *gradis = t.rad_gradis, *qcan = t.rad_qcan;  // qcan[l + 2*b]
    gradis[0] = gradis[1] = K(0.0);
#pragma unroll
    for (int k = 0; k < 6; k++) qcan[k] = K(0.0);
    R rho = t.air_rho[0];
    if (vlaiw > LAI_THRESH) {
      gradis[0] = DIV(DIV(K(4.0) * EMLEAF, CAPP * rho) * flpwb, tvrad) * extkd *
                  (DIV(K(1.0) - transb * transd, extkb + extkd) + DIV(transd - transb, extkb - extkd));
      gradis[1] = DIV(DIV(DIV(K(8.0) * EMLEAF, CAPP * rho) * flpwb, tvrad) * extkd * (K(1.0) - transd), extkd) -
                  gradis[0];
      qcan[4] = DIV((flws - flwv) * extkd * (transd - transb), extkb - extkd) +
                DIV((emair - EMLEAF) * extkd * flpwb * (K(1.0) - transd * transb), extkb + extkd);
      qcan[5] = (K(1.0) - transd) * (flws + t.met_fld[0] - K(2.0) * flwv) - qcan[4];
    }
    gradis[0] = t.air_cmolar[0] * gradis[0];
    gradis[1] = t.air_cmolar[0] * gradis[1];
    gradis[0] = MAX(K(1.0e-3), gradis[0]);
    gradis[1] = MAX(K(1.0e-3), gradis[1]);
    R cf1 = K(0.0), cf3 = K(0.0);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (sunlit_veg) {
        R kdm = t.rad_extkdm[b], kbm = t.rad_extkbm[b], fb = t.rad_fbeam[b];
        R rdf = t.rad_reffdf[b], rbm = t.rad_reffbm[b];
        R ckd = t.rad_cexpkdm[b], ckb = t.rad_cexpkbm[b];
        R tl = PV(veg_taul, b), rl = PV(veg_refl, b);
        cf1 = DIV(K(1.0) - transb * ckd, extkb + kdm);
        cf3 = DIV(K(1.0) - transb * ckb, extkb + kbm);
        R fsd = t.met_fsd[b];
        R tb = (DIV(K(1) - transb, extkb) - DIV(K(1) - p2(transb), extkb + extkb));
        qcan[0 + 2 * b] = fsd * ((K(1.0) - fb) * (K(1.0) - rdf) * kdm * cf1 + fb * (K(1.0) - rbm) * kbm * cf3 +
                                 fb * (K(1.0) - tl - rl) * extkb * tb);
        qcan[1 + 2 * b] = fsd * ((K(1.0) - fb) * (K(1.0) - rdf) * kdm * (DIV(K(1.0) - ckd, kdm) - cf1) +
                                 fb * (K(1.) - rbm) * kbm * (DIV(K(1.0) - ckb, kbm) - cf3) -
                                 fb * (K(1.0) - tl - rl) * extkb * tb);
      }
    }
    R *fsd = t.met_fsd;
    if (sunlit_veg) {
      t.rad_qssabs[0] =
          fsd[0] * (t.rad_fbeam[0] * (K(1.) - t.rad_reffbm[0]) * exp(-MIN(t.rad_extkbm[0] * vlaiw, K(20.))) +
                    (K(1.) - t.rad_fbeam[0]) * (K(1.) - t.rad_reffdf[0]) *
                        exp(-MIN(t.rad_extkdm[0] * vlaiw, K(20.)))) +
          fsd[1] * (t.rad_fbeam[1] * (K(1.) - t.rad_reffbm[1]) * t.rad_cexpkbm[1] +
                    (K(1.) - t.rad_fbeam[1]) * (K(1.) - t.rad_reffdf[1]) * t.rad_cexpkdm[1]);
      t.rad_scalex[0] = DIV(K(1.0) - transb * cf2n, extkb + extkn);
      t.rad_fvlai[0] = DIV(K(1.0) - transb, extkb);
      t.rad_fvlai[1] = vlaiw - t.rad_fvlai[0];
    } else {
      t.rad_qssabs[0] = (K(1.0) - t.ssnow_albsoilsn[0]) * fsd[0] + (K(1.0) - t.ssnow_albsoilsn[1]) * fsd[1];
      t.rad_scalex[0] = K(0.0);
      t.rad_fvlai[0] = K(0.0);
      t.rad_fvlai[1] = vlaiw;
    }
    t.rad_scalex[1] = DIV(K(1.0) - cf2n, extkn) - t.rad_scalex[0];
#pragma unroll
    for (int l = 0; l < 2; l++) t.rad_rniso[l] = qcan[l + 0] + qcan[l + 2] + qcan[l + 4];
  }

  // src/science/canopy/cbl_friction_vel.F90:112-166
  // psim and psis: the reference blends the stable and unstable forms as
  // z*stable + (1-z)*unstable with z = 0.5 + SIGN(0.5, zeta), which is 0 or 1;
  // both forms are finite for the clamped zeta, so the blend returns the
  // selected form exactly and only that form is evaluated
  CBM_HD static bool stable(R zeta) { return K(0.5) + SIGN(K(0.5), zeta) > K(0.5); }
  CBM_HD static R psim_stable(R zeta) {
    const R a_ = K(1.0), b = K(0.667), xc = K(5.0), d = K(0.35);
    return -a_ * zeta - b * (zeta - DIV(xc, d)) * exp(-d * zeta) - DIV(b * xc, d);
  }
  CBM_HD static R psim_unstable(R zeta) {
    const R gu = K(16.0);
    R x = root4(K(1.0) + gu * fabs(zeta));
    return log((K(1.0) + x * x) * p2(K(1.0) + x) / K(8)) - K(2.0) * atan(x) + PI_C * K(0.5);
  }
  CBM_HD static R psim(R zeta) { return stable(zeta) ? psim_stable(zeta) : psim_unstable(zeta); }

  // src/science/canopy/cbl_friction_vel.F90:168-221
  CBM_HD static R psis_stable(R zeta) {
    const R a_ = K(1.0), b = K(0.667), c = K(5.0), d = K(0.35);
    R stzeta = MAX(K(0.), zeta);
    return -pow1p5(K(1.) + K(2.) / K(3.) * a_ * stzeta) - b * (stzeta - DIV(c, d)) * exp(-d * stzeta) - DIV(b * c, d) +
           K(1.);
  }
  CBM_HD static R psis_unstable(R zeta) {
    const R gu = K(16.0);
    R y = sqrt(K(1.0) + gu * fabs(zeta));
    return K(2.0) * log((K(1) + y) * K(0.5));
  }
  CBM_HD static R psis(R zeta) { return stable(zeta) ? psis_stable(zeta) : psis_unstable(zeta); }

  // src/science/canopy/cbl_dryLeaf.F90:779-877
  // (c4ca = 4 convex alpha, r2 = recip(2 convex))
  CBM_HD static R ej3x(R parx, R alpha, R convex, R x, R c4ca, R r2) {
    return MAX(K(0.0), K(0.25) * DIVR(alpha * parx + x - sqrt(p2(alpha * parx + x) - c4ca * parx * x),
                                   K(2.0) * convex, r2));
  }
  CBM_HD static R ej4x(R parx, R alpha, R convex, R x, R c4ca, R r2) {
    return MAX(K(0.0), DIVR(alpha * parx + x - sqrt(p2(alpha * parx + x) - c4ca * parx * x),
                            K(2.0) * convex, r2));
  }
  CBM_HD static R xvcmxt4(R x) {
    return DIV(exp2(K(0.1) * x - K(2.5)), (K(1.0) + exp(K(0.3) * (K(13.0) - x))) * (K(1.0) + exp(K(0.3) * (x - K(36.0)))));
  }
  CBM_HD static R xvcmxt3(R x) {
    const R EHaVc = K(73637.0), EHdVc = K(149252.0), EntropVc = K(486.0), xVccoef = K(1.17461);
    R num = xVccoef * exp(DIV(EHaVc, RGAS * TREFK) * (K(1.) - DIV(TREFK, x)));
    R den = K(1.0) + exp(DIV(EntropVc * x - EHdVc, RGAS * x));
    return MAX(K(0.0), DIV(num, den));
  }
  CBM_HD static R xejmxt3(R x) {
    const R EHaJx = K(50300.0), EHdJx = K(152044.0), EntropJx = K(495.0), xjxcoef = K(1.16715);
    R num = xjxcoef * exp(DIV(EHaJx, RGAS * TREFK) * (K(1.) - DIV(TREFK, x)));
    R den = K(1.0) + exp(DIV(EntropJx * x - EHdJx, RGAS * x));
    return MAX(K(0.0), DIV(num, den));
  }

  // The larger root of coef2 z^2 + coef1 z + coef0 = 0 as the reference
  // takes it, (-coef1 + sqrt(max(0, delcx))) / (2 coef2) with delcx =
  // coef1^2 - 4 coef0 coef2 (cbl_photosynthesis.F90:107-111, 157-161,
  // 202-206).  The reference holds these coefficients in REAL(r_2) (FP64,
  // :36-38).  In FP32 (the mixed path) the sum -coef1 + sqrt(delcx) cancels
  // when coef1 > 0 and loses the root's digits, so there the equal
  // 2 coef0 / (-coef1 - sqrt(delcx)) is taken, which keeps them: the canopy's
  // GPP then stays as close to FP64 as the reference's own shipped build
  // does.  FP64 keeps the reference's form.
  CBM_HD static R larger_root(R coef2z, R coef1z, R coef0z) {
    const R delcxz = p2(coef1z) - K(4.0) * coef0z * coef2z;
    const R s = sqrt(MAX(K(0.0), delcxz));
    if constexpr (sizeof(R) == 4) {
      const bool b = coef1z > K(0.0);
      const R d = (b ? -s : s) - coef1z;
      return DIV(b ? K(2.0) * coef0z : d, b ? d : K(2.0) * coef2z);
    }
    const bool linear = !(fabs(coef2z) >= K(1.0e-9));
    return DIV(linear ? -coef0z : -coef1z + s, linear ? coef1z : K(2.0) * coef2z);
  }

  // src/science/canopy/cbl_photosynthesis.F90:10-226, one leaf.  The three
  // limits' quadratics are solved side by side, so that their chains of
  // square roots and quotients overlap.  A coefficient of z^2 too small for
  // the root (none with the shipped parameters) takes the reference's linear
  // form: in FP64, whose one wave per SIMD waits on those chains, by selected
  // operands of the one quotient, which keeps both leaves in one block (a
  // day of 262,144 tiles 17.1 against 17.9 ms); in FP32, bound by issue, in
  // a branch for the three (a day of 1,048,576 tiles 19.8 against 20.8 ms).
  CBM_HD static R photosynthesis_leaf(R csxz, R cx1z, R cx2z, R gswminz, R rdxz, R vcmxt3z,
                                          R vcmxt4z, R vx3z, R vx4z, R gs_coeffz, R fwsoilz) {
    const R effc4 = K(4000.0);
    R gf = DIV(gswminz * fwsoilz, RGSWC);
    R coef0[3], coef1[3], coef2[3];
    coef2[0] = gf + gs_coeffz * (vcmxt3z - (rdxz - vcmxt4z));
    coef1[0] = (K(1.0) - csxz * gs_coeffz) * (vcmxt3z + vcmxt4z - rdxz) + DIV(gswminz * fwsoilz, RGSWC) * (cx1z - csxz) -
               gs_coeffz * (vcmxt3z * cx2z / K(2.0) + cx1z * (rdxz - vcmxt4z));
    coef0[0] = -(K(1.0) - csxz * gs_coeffz) * (vcmxt3z * cx2z / K(2.0) + cx1z * (rdxz - vcmxt4z)) -
               DIV(gswminz * fwsoilz, RGSWC) * cx1z * csxz;
    coef2[1] = gf + gs_coeffz * (vx3z - (rdxz - vx4z));
    coef1[1] = (K(1.0) - csxz * gs_coeffz) * (vx3z + vx4z - rdxz) + DIV(gswminz * fwsoilz, RGSWC) * (cx2z - csxz) -
               gs_coeffz * (vx3z * cx2z / K(2.0) + cx2z * (rdxz - vx4z));
    coef0[1] = -(K(1.0) - csxz * gs_coeffz) * (vx3z * cx2z / K(2.0) + cx2z * (rdxz - vx4z)) -
               DIV(gswminz * fwsoilz, RGSWC) * cx2z * csxz;
    coef2[2] = gs_coeffz;
    coef1[2] = gf + gs_coeffz * (rdxz - K(0.5) * vcmxt3z) + effc4 * vcmxt4z - gs_coeffz * csxz * effc4 * vcmxt4z;
    coef0[2] = -DIV(gswminz * fwsoilz, RGSWC) * csxz * effc4 * vcmxt4z + DIV((rdxz - K(0.5) * vcmxt3z) * gswminz * fwsoilz, RGSWC);
    R z[3];
#pragma unroll
    for (int q = 0; q < 3; q++) z[q] = larger_root(coef2[q], coef1[q], coef0[q]);
    // a limit whose coefficients give neither form keeps the reference's initial
    // value: both too small, or (FP64) NaN (in coef1, whose terms hold the
    // factors of coef2, so that two compares a limit tell)
    bool solved[3];
#pragma unroll
    for (int q = 0; q < 3; q++)
      solved[q] = sizeof(R) == 4 || fabs(coef2[q]) >= K(1.0e-9) || fabs(coef1[q]) >= K(1.0e-9);
    if (sizeof(R) == 4 && (fabs(coef2[0]) < K(1.0e-9) || fabs(coef2[1]) < K(1.0e-9) || fabs(coef2[2]) < K(1.0e-9))) {
#pragma unroll
      for (int q = 0; q < 3; q++)
        if (fabs(coef2[q]) < K(1.0e-9)) {
          z[q] = DIV(-coef0[q], coef1[q]);
          solved[q] = fabs(coef1[q]) >= K(1.0e-9);
        }
    }
    R ciz = MAX(K(0.0), z[0]);
    R anrubiscoz = DIV(vcmxt3z * (ciz - cx2z / K(2.0)), ciz + cx1z) + vcmxt4z - rdxz;
    anrubiscoz = solved[0] ? anrubiscoz : K(0.0);
    ciz = MAX(K(0.0), z[1]);
    R anrubpz = DIV(vx3z * (ciz - cx2z / K(2.0)), ciz + cx2z) + vx4z - rdxz;
    anrubpz = solved[1] ? anrubpz : K(99999.0);
    const R ansinkz = solved[2] ? z[2] : fabs(coef1[2]) < K(1.0e-9) ? K(99999.0) : K(0.0);
    return MIN(MIN(anrubiscoz, anrubpz), ansinkz);
  }

  // src/science/soilsnow/cbl_remove_trans.F90:43-93.  The canopy iteration's
  // REAL(r_2) quantities (transpiration per layer, fevc, fess, dgdtg) are
  // computed in the step's working precision R: FP64 in the plain path, FP32
  // in the mixed path, whose FP64 is kept to the tridiagonal solves and the
  // balance accumulators.  avail[k], the water layer k can give
  // (MAX(0, wbliq - 1.1 swilt) zse 1000), does not change during the canopy
  // iteration and is computed once per step (define_canopy).
  CBM_HD void transp_soil_water(R fevc, const R *avail, R *evapfbl) {
    R diff_prev = K(0.0);
#pragma unroll
    for (int k = 0; k < MS; k++) {
      R xx = DIV(fevc * (R)a.dels, HL) * PV(veg_froot, k) + diff_prev;
      R xxd = xx - avail[k];
      if (xxd > K(0.0)) {
        evapfbl[k] = avail[k];
        diff_prev = xxd;
      } else {
        evapfbl[k] = xx;
        diff_prev = K(0.0);
      }
    }
  }

  // working variables define_canopy shares with dryLeaf and wetLeaf
  struct Can {
    R cansat, dsx, fwsoil, tlfx, tlfy, ecy, hcy, rny;
    R gbhu[2], gbhf[2], csx[2], ghwet;
    R sum_rad_rniso, sum_rad_gradis;
    R avail[MS];   // water each soil layer can give to transpiration, mm
  };

  // src/science/canopy/cbl_dryLeaf.F90:10-666
  CBM_HD void dryLeaf(Can &c, int iter) {
    const R jtomol = K(4.6e-6);
    R dels = (R)a.dels;
    R vlaiw = t.canopy_vlaiw[0];
    R rlam = t.air_rlam[0];
    R gs_coeff[2] = {K(0.0), K(0.0)};
    if (iter == 1) {
      // fwsoil_calc_std, src/science/canopy/cbl_fwsoil.F90:13-38
      R s = K(0.0);
#pragma unroll
      for (int k = 0; k < MS; k++) {
        const R swilt = (R)PV(soil_swilt_vec, k);
        R r = DIV((R)t.ssnow_wbliq[k] - swilt, (R)PV(soil_sfc_vec, k) - swilt);
        R term = PV(veg_froot, k) * MAX(K(1.0e-9), MIN(K(1.0), r));
        s = (k == 0) ? term : s + term;
      }
      R rwater = MAX(K(1.0e-9), s);
      c.fwsoil = MAX(K(1.0e-9), MIN(K(1.0), PV(veg_vbeta, 0) * rwater));
      t.canopy_fwsoil[0] = c.fwsoil;
    }
    R fwsoil = c.fwsoil;
    R gswmin[2];
    R vgswmin = PV(veg_gswmin, 0);
    gswmin[0] = MAX(K(1.e-6), t.rad_scalex[0] * vgswmin);
    gswmin[1] = MAX(K(1.e-6), t.rad_scalex[1] * vgswmin);
    R gh[2] = {K(1.0e-3), K(1.0e-3)}, ghr[2] = {K(1.0e-3), K(1.0e-3)};
    R rdx[2] = {K(0.0), K(0.0)}, anx[2] = {K(0.0), K(0.0)}, an_y[2] = {K(0.0), K(0.0)},
      rdy[2] = {K(0.0), K(0.0)};
    R rnx = c.sum_rad_rniso, abs_deltlf = K(999.0);
    R hcx = K(0.0), ecx = c.sum_rad_rniso;
    c.hcy = K(0.0);
    R tlfxx = c.tlfx;
    R psycst[2] = {t.air_psyc[0], t.air_psyc[0]};
    R vcmxt3[2] = {K(0), K(0)}, vcmxt4[2] = {K(0), K(0)}, vx3[2] = {K(0), K(0)}, vx4[2] = {K(0), K(0)};
    R cx1 = K(0.0), cx2 = K(0.0), deltlf = K(0.0);
    // canopy%fevc and ssnow%evapfbl while the passes run; stored at the end
    R fevc = K(0.0), evapfbl[MS], oldevapfbl[MS];
#pragma unroll
    for (int k = 0; k < MS; k++) evapfbl[k] = K(0.0);
    c.ghwet = K(1.0e-3);
    t.canopy_fevw[0] = K(0.0);
    t.canopy_fhvw[0] = K(0.0);
    R sum_gbh = (c.gbhu[0] + c.gbhf[0]) + (c.gbhu[1] + c.gbhf[1]);
    if (vlaiw <= LAI_THRESH) {
      rnx = K(0.0);
      ecx = K(0.0);
      c.ecy = ecx;
      abs_deltlf = K(0.0);
      c.rny = rnx;
    }
    R deltlfy = abs_deltlf;
    const R tvair = t.met_tvair[0], tk = t.met_tk[0];
    const R fvl0 = t.rad_fvlai[0], fvl1 = t.rad_fvlai[1];
    const bool leaves = fvl0 + fvl1 > LAI_THRESH;
    // whether the class has C3 and C4 leaves; in FP64 also set where the terms
    // of the absent ones are not zero: a share of zero times NaN or infinity
    bool c3 = true, c4 = PV(veg_frac4, 0) != K(0.0);
    if constexpr (sizeof(R) == 8) {
      const R convex = fabs(PV(veg_convex, 0));
      const bool odd = !(fabs(PV(veg_vcmax, 0)) < K(1e30) && fabs(PV(veg_ejmax, 0)) < K(1e30) &&
                         fabs(PV(veg_alpha, 0)) < K(1e30) && convex > K(0.0) && convex < K(1e30));
      c3 = PV(veg_frac4, 0) != K(1.0) || odd;
      c4 = c4 || odd;
    }
    // the reference's fixed count of 20 passes.  The hybrid polishes the
    // start of a sunlit leaf-bearing tile with a.max_passes passes and then
    // checks it by its leaf energy-balance residual: the leaf
    // sensible-plus-radiative conductance times the temperature change the
    // last pass still made, beyond the 0.1 K the reference's own convergence
    // test accepts, cr (ghr1 + ghr2) (|dT| - 0.1 K).  Within a.resid_max
    // (W/m2) the tile stops there.  Otherwise it falls back to the
    // reference's iteration for the rest of the step: the passes go on from
    // where they are, with the reference's damping, up to its 20.  (From the
    // reference's own start -- the NITER passes after the first, or a run
    // without the network -- the capped passes are the reference's own, so
    // the fallback is the reference's iteration exactly.  Starting the first
    // NITER pass again from the reference's start instead was measured:
    // 0.547 against 0.523 ms per step at 1,048,576 tiles, and no more
    // accurate.)  Every other tile runs the reference's iteration.
    // (one copy of the body: the hybrid's first passes would otherwise be
    // peeled off, 8% more instructions)
    for (int k = 1; k <= 20; k++) {
      bool active = (vlaiw > LAI_THRESH && abs_deltlf > K(0.1));
      if constexpr (MODE == MODE_HYBRID) {
        if (capped && active && k == a.max_passes + 1) {
          const float r = (float)(CAPP * RMAIR * (ghr[0] + ghr[1]) * (abs_deltlf - K(0.1)));
          if (r <= a.resid_max) {
            active = false;
          } else {
            fell_back = true;
            capped = false;
          }
        }
      }
      // a tile that has converged keeps every value: the remaining passes of
      // the reference's fixed-count loop change nothing for it
      if (!active && k > 1) break;
      anx[0] = anx[1] = K(0.0);
      if (active) {
        npass++;
        R tlfx = c.tlfx;
        R dleaf = PV(veg_dleaf, 0);
        c.ghwet = K(2.0) * sum_gbh;
        R gras = MAX(K(1.0e-6), K(1.595E8) * fabs(tlfx - tvair) * derived(VX_dleaf3));
        R g25 = root4(gras);
        const R rdleaf = derived(VX_rdleaf);
        c.gbhf[0] = DIVR(fvl0 * t.air_cmolar[0] * K(0.5) * DHEAT * (g25), dleaf, rdleaf);
        c.gbhf[1] = DIVR(fvl1 * t.air_cmolar[0] * K(0.5) * DHEAT * (g25), dleaf, rdleaf);
        c.gbhf[0] = MAX(K(1.e-6), c.gbhf[0]);
        c.gbhf[1] = MAX(K(1.e-6), c.gbhf[1]);
#pragma unroll
        for (int l = 0; l < 2; l++) {
          gh[l] = K(2.0) * (c.gbhu[l] + c.gbhf[l]);
          ghr[l] = t.rad_gradis[l] + gh[l];
        }
        R frac4 = PV(veg_frac4, 0), vcmax = PV(veg_vcmax, 0);
        R tdiff = tlfx - TREFK;
        R conkct = PV(veg_conkc0, 0) * exp(derived(VX_ekc) * (K(1.0) - DIV(TREFK, tlfx)));
        R conkot = PV(veg_conko0, 0) * exp(derived(VX_eko) * (K(1.0) - DIV(TREFK, tlfx)));
        tlfxx = tlfx;
        cx1 = conkct * (K(1.0) + DIV(K(0.21), conkot));
        cx2 = K(2.0) * GAM0 * (K(1.0) + GAM1 * tdiff + GAM2 * tdiff * tdiff);
        R alpha = PV(veg_alpha, 0), convex = PV(veg_convex, 0);
        const R c4ca = derived(VX_c4ca), r2 = derived(VX_r2convex);
        R q0 = t.rad_qcan[0], q1 = t.rad_qcan[1];
        // the C3 and the C4 terms each carry the class's share as a factor:
        // without one they are zero, and their exponentials and roots are
        // left out (in FP32 the C4 terms only: the branch around the C3 terms
        // waits for the class table and costs more than it saves).  A leaf
        // iterate near or below 0 K, where the exponentials overflow, keeps
        // them, and with them the reference's NaN
        if constexpr (sizeof(R) == 8) {
          const bool hot = !(tlfx >= K(64.0) && tlfx < K(1024.0));
          c3 = c3 || hot;
          c4 = c4 || hot;
        }
        if (sizeof(R) == 4 || c3) {
          R temp = xvcmxt3(tlfx) * vcmax * (K(1.0) - frac4);
          vcmxt3[0] = t.rad_scalex[0] * temp;
          vcmxt3[1] = t.rad_scalex[1] * temp;
          temp = xejmxt3(tlfx) * PV(veg_ejmax, 0) * (K(1.0) - frac4);
          R ejmxt3_0 = t.rad_scalex[0] * temp, ejmxt3_1 = t.rad_scalex[1] * temp;
          vx3[0] = ej3x(q0 * jtomol * (K(1.0) - frac4), alpha, convex, ejmxt3_0, c4ca, r2);
          vx3[1] = ej3x(q1 * jtomol * (K(1.0) - frac4), alpha, convex, ejmxt3_1, c4ca, r2);
        }
        if (c4) {
          R temp = xvcmxt4(tlfx - TFRZ) * vcmax * frac4;
          vcmxt4[0] = t.rad_scalex[0] * temp;
          vcmxt4[1] = t.rad_scalex[1] * temp;
          vx4[0] = ej4x(q0 * jtomol * frac4, alpha, convex, vcmxt4[0], c4ca, r2);
          vx4[1] = ej4x(q1 * jtomol * frac4, alpha, convex, vcmxt4[1], c4ca, r2);
        }
        R cfrd = PV(veg_cfrd, 0);
        rdx[0] = (cfrd * vcmxt3[0] + cfrd * vcmxt4[0]);
        rdx[1] = (cfrd * vcmxt3[1] + cfrd * vcmxt4[1]);
        R a1 = DIV(PV(veg_a1gs, 0), K(1.0) + DIVR(c.dsx, PV(veg_d0gs, 0), derived(VX_rd0gs)));
        gs_coeff[0] = DIV(fwsoil, c.csx[0] - K(0.0)) * a1;
        gs_coeff[1] = DIV(fwsoil, c.csx[1] - K(0.0)) * a1;
        // one leaf's assimilation, leaf-surface CO2 and conductances; `has`:
        // the leaf class has leaves (else its values stay)
        auto leaf = [&](int l, bool has) {
          const R an = photosynthesis_leaf(c.csx[l], cx1, cx2, gswmin[l], rdx[l], vcmxt3[l], vcmxt4[l], vx3[l],
                                           vx4[l], gs_coeff[l], fwsoil);
          anx[l] = has && leaves ? an : K(0.0);
          R cs = t.met_ca[0] - DIV(RGBWC * anx[l], c.gbhu[l] + c.gbhf[l]);
          c.csx[l] = has ? MAX(K(1.0e-4), cs) : c.csx[l];
          const R gsw = MAX(K(1.e-3), gswmin[l] * fwsoil + MAX(K(0.0), RGSWC * gs_coeff[l] * anx[l]));
          t.canopy_gswx[l] = has ? gsw : t.canopy_gswx[l];
          R gw = DIV(K(1.0), DIV(K(1.0), t.canopy_gswx[l]) + DIV(K(1.0), K(1.075) * (c.gbhu[l] + c.gbhf[l])));
          gw = MAX(gw, K(0.00001));
          const R ps = t.air_psyc[0] * DIV(ghr[l], gw);
          psycst[l] = has ? ps : psycst[l];
        };
        // sunlit and shaded leaves side by side by day, shaded leaves alone
        // without light
        if (fvl0 > LAI_THRESH) {
          leaf(0, true);
          leaf(1, fvl1 > LAI_THRESH);
        } else if (fvl1 > LAI_THRESH) {
          leaf(1, true);
        }
        R dsatdk = t.air_dsatdk[0], dtv = tvair - tk;
        R cr = CAPP * RMAIR;
        ecx = DIV(dsatdk * (t.rad_rniso[0] - cr * dtv * t.rad_gradis[0]) + cr * t.met_dva[0] * ghr[0],
                  dsatdk + psycst[0]) +
              DIV(dsatdk * (t.rad_rniso[1] - cr * dtv * t.rad_gradis[1]) + cr * t.met_dva[0] * ghr[1],
                  dsatdk + psycst[1]);
        R fwet = t.canopy_fwet[0];
        R local_fevc = (K(1.0) - fwet) * ecx;
        if (local_fevc > K(0.0)) {
          transp_soil_water(local_fevc, c.avail, evapfbl);
          R s = evapfbl[0];
#pragma unroll
          for (int q = 1; q < MS; q++) s = s + evapfbl[q];
          fevc = DIV(s * rlam, (R)a.dels);
          ecx = DIV(fevc, K(1.0) - fwet);
        }
        hcx = DIV((c.sum_rad_rniso - ecx - cr * dtv * c.sum_rad_gradis) * (gh[0] + gh[1]), ghr[0] + ghr[1]);
        c.tlfx = tvair + DIV(hcx, cr * (gh[0] + gh[1]));
        rnx = c.sum_rad_rniso - cr * (c.tlfx - tk) * c.sum_rad_gradis;
        c.dsx = t.met_dva[0] + dsatdk * (c.tlfx - tvair);
        c.dsx = MAX(c.dsx, K(0.0));
        deltlf = tlfxx - c.tlfx;
        abs_deltlf = fabs(deltlf);
      }
      if (abs_deltlf < fabs(deltlfy)) {
        deltlfy = deltlf;
        c.tlfy = c.tlfx;
        c.rny = rnx;
        c.hcy = hcx;
        c.ecy = ecx;
        rdy[0] = rdx[0];
        rdy[1] = rdx[1];
        an_y[0] = anx[0];
        an_y[1] = anx[1];
#pragma unroll
        for (int q = 0; q < MS; q++) oldevapfbl[q] = evapfbl[q];
      }
      if (abs_deltlf > K(0.1)) {
        R w = K(0.5) * DIV((R)(k - 5 > 0 ? k - 5 : 0), (R)k - K(4.9999));
        c.tlfx = w * tlfxx + (K(1.0) - w) * c.tlfx;
      }
      if (k == 1) {
        c.tlfy = c.tlfx;
        c.rny = rnx;
        c.hcy = hcx;
        c.ecy = ecx;
        rdy[0] = rdx[0];
        rdy[1] = rdx[1];
        an_y[0] = anx[0];
        an_y[1] = anx[1];
#pragma unroll
        for (int q = 0; q < MS; q++) oldevapfbl[q] = evapfbl[q];
      }
    }
    R fwet = t.canopy_fwet[0];
    fevc = (K(1.0) - fwet) * c.ecy;
    if (c.ecy > K(0.0) && fwet < K(1.0)) {
      if (fabs(c.ecy - ecx) > K(1.0e-6)) {
        R s = oldevapfbl[0];
#pragma unroll
        for (int q = 1; q < MS; q++) s = s + oldevapfbl[q];
        if (!(fabs(fevc - DIV(s * rlam, (R)a.dels)) > K(1.0e-4))) {
#pragma unroll
          for (int q = 0; q < MS; q++) evapfbl[q] = oldevapfbl[q];
        }
      }
    }
    t.canopy_fevc[0] = fevc;
#pragma unroll
    for (int q = 0; q < MS; q++) t.ssnow_evapfbl[q] = evapfbl[q];
    t.canopy_frday[0] = K(12.0) * (rdy[0] + rdy[1]);
    t.canopy_fpn[0] = MIN(-K(12.0) * (an_y[0] + an_y[1]), t.canopy_frday[0]);
  }

  // src/science/canopy/cbl_wetleaf.F90:9-111
  CBM_HD void wetLeaf(Can &c) {
    R dels = (R)a.dels;
    c.ghwet = K(1.0e-3);
    R gwwet, ghrwet;
    t.canopy_fevw[0] = K(0.0);
    t.canopy_fhvw[0] = K(0.0);
    R sum_gbh = (c.gbhu[0] + c.gbhf[0]) + (c.gbhu[1] + c.gbhf[1]);
    if (t.canopy_vlaiw[0] > LAI_THRESH) {
      R rlam = t.air_rlam[0], dsatdk = t.air_dsatdk[0], psyc = t.air_psyc[0];
      R srn = c.sum_rad_rniso, sg = c.sum_rad_gradis, fwet = t.canopy_fwet[0];
      c.ghwet = K(2.0) * sum_gbh;
      gwwet = K(1.075) * sum_gbh;
      ghrwet = sg + c.ghwet;
      R ccfevw = MIN(DIV(t.canopy_cansto[0] * rlam, dels), DIV(K(2.0), DIV(K(1440.0), DIV(dels, K(60.0)))) * rlam);
      R dtv = t.met_tvair[0] - t.met_tk[0];
      R cr = CAPP * RMAIR;
      R num = dsatdk * (srn - cr * dtv * sg) + cr * t.met_dva[0] * ghrwet;
      R den = dsatdk + DIV(psyc * ghrwet, gwwet);
      t.canopy_fevw[0] = MIN(DIV(fwet * num, den), ccfevw);
      t.canopy_fevw_pot[0] = DIV(num, den);
      t.canopy_fhvw[0] = fwet * (srn - cr * (c.tlfy - t.met_tk[0]) * sg) - t.canopy_fevw[0];
    }
  }

  // src/science/canopy/cbl_pot_evap_snow.F90:79-167 (HDM)
  CBM_HD R humidity_deficit_method(R dq, R dqu) {
    if (t.ssnow_snowd[0] > K(1.0) || t.ssnow_tgg[0] == TFRZ) {
      dq = MAX(-K(0.1e-3), dq);
      dqu = MAX(-K(0.1e-3), dqu);
    }
    (void)dqu;
    return DIV(t.air_rho[0] * t.air_rlam[0] * dq, t.ssnow_rtsoil[0]);
  }

  // src/science/canopy/cbl_latent_heat.F90:15-285
  CBM_HD void latent_heat_flux() {
    R dels = (R)a.dels;
    R potev = t.ssnow_potev[0], rlam = t.air_rlam[0], snowd = t.ssnow_snowd[0];
    if (potev < K(0.)) t.ssnow_wetfac[0] = K(1.0);
    R wetfac = t.ssnow_wetfac[0];
    R fess = wetfac * potev;
    R pudsto = t.ssnow_pudsto[0];
    R pwet = MAX(K(0.), MIN(K(0.2), DIV(pudsto, MAX(K(1.), (R)PV(ssnow_pudsmx, 0)))));
    fess = fess * (K(1.) - pwet);
    R frescale = DIV((R)a.zse[0] * DENSITY_LIQ * rlam, dels);
    if (snowd < K(0.1) && fess > K(0.)) {
      R flower = (R)t.ssnow_wb[0] - PV(soil_swilt, 0) / K(2.0);
      R fupper = MAX(K(0.), flower * frescale - DIV((R)t.ssnow_evapfbl[0] * rlam, dels));
      fess = MIN(fess, fupper);
      fupper = (R)(t.ssnow_wb[0] - DIV(t.ssnow_wbice[0], (double)FROZEN_LIMIT)) * frescale;
      fupper = MAX(fupper, K(0.));
      fess = MIN(fess, fupper);
    }
    R cls = K(1.);
    if (snowd >= K(0.1)) {
      cls = K(1.1335);
      fess = cls * potev;
    }
    if (snowd < K(0.1) && potev < K(0.) && t.ssnow_tss[0] < TFRZ) {
      cls = K(1.1335);
      fess = cls * potev;
    }
    if (snowd >= K(0.1) && potev > K(0.)) {
      cls = K(1.1335);
      fess = MIN((wetfac * potev) * cls, DIV(snowd, dels) * rlam * cls);
    }
    t.ssnow_cls[0] = cls;
    R fesp = MIN(DIV(pudsto, dels) * rlam, MAX(pwet * potev, K(0.)));
    t.canopy_fess[0] = fess;
    t.canopy_fesp[0] = fesp;
    t.canopy_fes[0] = fess + fesp;
  }

  // src/science/canopy/cbl_within_canopy.F90:10-159
  CBM_HD void within_canopy(Can &c, R rt0, R &qstvair) {
    R cmolar = t.air_cmolar[0];
    R rrbw = DIV((c.gbhu[0] + c.gbhf[0]) + (c.gbhu[1] + c.gbhf[1]), cmolar);
    R rrsw = DIV(t.canopy_gswx[0] + t.canopy_gswx[1], cmolar);
    R fix_eqn = DIV(t.ssnow_cls[0] * rt0, rt0 + K(0.0));
    if (t.ssnow_potev[0] > K(0.)) fix_eqn = fix_eqn * t.ssnow_wetfac[0];
    R fix_eqn2 = DIV(rt0, rt0 + K(0.0));
    if (PV(veg_meth, 0) > K(0) && t.canopy_vlaiw[0] > LAI_THRESH && t.rough_hruff[0] > t.rough_z0soilsn[0]) {
      R epsi = t.air_epsi[0], rt1 = t.rough_rt1[0], rlam = t.air_rlam[0];
      R rho = t.air_rho[0];
      R e1 = (K(1.) + epsi) * rrsw + rrbw;
      R dmah = (rt0 + fix_eqn2 * rt1) * e1 + epsi * (rt0 * rt1) * (rrbw * rrsw);
      R dmbh = DIV(-rlam, CAPP) * (rt0 * rt1) * (rrbw * rrsw);
      R dmch = DIV(e1 * rt0 * rt1 * (t.canopy_fhv[0] + t.canopy_fhs[0]), rho * CAPP);
      R dmae = DIV(-epsi * CAPP, rlam) * (rt0 * rt1) * (rrbw * rrsw);
      R dmbe = (rt0 + fix_eqn * rt1) * e1 + (rt0 * rt1) * (rrbw * rrsw);
      R dmce = DIV(e1 * rt0 * rt1 * ((R)t.canopy_fev[0] + DIV((R)t.canopy_fes[0], t.ssnow_cls[0])), rho * rlam);
      R tk = t.met_tk[0], tss = t.ssnow_tss[0];
      R det = dmah * dmbe - dmae * dmbh + K(1.0e-12);
      R tvair = tk + DIV(dmbe * dmch - dmbh * dmce, det);
      R lo = MIN(tss, tk) - K(5.0), hi = MAX(tss, tk) + K(5.0);
      tvair = MAX(tvair, lo);
      tvair = MIN(tvair, hi);
      t.met_tvair[0] = tvair;
      R qv = t.met_qv[0];
      R qvair = qv + DIV(dmah * dmce - dmae * dmch, det);
      qvair = MAX(K(0.0), qvair);
      lo = MIN(t.ssnow_qstss[0], qv);
      hi = MAX(t.ssnow_qstss[0], qv);
      qvair = MAX(qvair, lo);
      qvair = MIN(qvair, hi);
      t.met_qvair[0] = qvair;
      qstvair = qsatfjh(tvair - TFRZ, t.met_pmb[0]);
      t.met_dva[0] = DIV((qstvair - qvair) * RMAIR, RMH2O) * t.met_pmb[0] * K(100.);
    }
  }

  // src/science/canopy/cable_canopy.F90:10-1048
  template <class Settled>
  CBM_HD void define_canopy(bool sunlit_veg, Settled &&settled) {
    Can c;
    R dels = (R)a.dels;
    R vlaiw = t.canopy_vlaiw[0];
    bool veg = vlaiw > LAI_THRESH;
    t.canopy_cansto[0] = t.canopy_oldcansto[0];
    c.cansat = PV(veg_canst1, 0) * vlaiw;
    {  // Surf_wetness_fact, src/science/canopy/cbl_SurfaceWetness.F90:10-79
      R precip = t.met_precip[0], psn = t.met_precip_sn[0];
      R upper = DIV(K(4.0) * MIN(dels, K(1800.0)), K(60.0) * K(1440.0));
      R ftemp = MIN(precip - psn, upper);
      R lower = c.cansat - t.canopy_cansto[0];
      upper = MAX(lower, K(0.0));
      R wcint = (ftemp > K(0.0) && t.met_tk[0] > TFRZ) ? MIN(upper, ftemp) : K(0.0);
      t.canopy_wcint[0] = wcint;
      t.canopy_through[0] = psn + MIN(precip - psn, MAX(K(0.0), precip - psn - wcint));
      t.canopy_cansto[0] = t.canopy_cansto[0] + wcint;
      t.canopy_fwet[0] = MAX(K(0.0), MIN(K(0.9), DIV(K(0.8) * t.canopy_cansto[0], MAX(c.cansat, K(0.01)))));
      t.ssnow_satfrac[0] = 1.0e-8;
      t.ssnow_rh_srf[0] = 1.0;
      // initialize_wetfac, src/science/canopy/cbl_init_wetfac_mod.F90:9-116
      R swilt = PV(soil_swilt, 0);
      R wilting_pt = swilt / K(2.0);
      R num = (R)t.ssnow_wb[0] - wilting_pt;
      R den = PV(soil_sfc, 0) - wilting_pt;
      den = MAX(K(0.0830), den);
      R wf = DIV(num, den);
      wf = MIN(K(1.0), wf);
      wf = MAX(K(0.0), wf);
      if (t.ssnow_wbice[0] > 0.0) {
        R ice_ratio = p2((R)(DIV(t.ssnow_wbice[0], t.ssnow_wb[0])));
        R ice_factor = K(1.0) - MIN(K(0.2), ice_ratio);
        ice_factor = MAX(K(0.5), ice_factor);
        wf = wf * ice_factor;
      }
      if (t.ssnow_snowd[0] > K(0.1)) wf = K(0.9);
      if (t.veg_iveg[0] == LAKES) {
        if (t.met_tk[0] >= TFRZ + K(5.)) wf = K(1.0);
        if (t.met_tk[0] < TFRZ + K(5.)) wf = K(0.7);
      }
      t.ssnow_wetfac[0] = K(0.5) * (wf + t.ssnow_owetfac[0]);
    }
    t.canopy_fevw_pot[0] = K(0.0);
    t.canopy_gswx[0] = t.canopy_gswx[1] = K(1e-3);
    c.gbhf[0] = c.gbhf[1] = K(1e-3);
    c.gbhu[0] = c.gbhu[1] = K(1e-3);
#pragma unroll
    for (int k = 0; k < MS; k++) t.ssnow_evapfbl[k] = 0.0, t.ssnow_rex[k] = 0.0;
    // the water each soil layer can give to transpiration this step
#pragma unroll
    for (int k = 0; k < MS; k++)
      c.avail[k] = (R)(MAX(0.0, t.ssnow_wbliq[k] - 1.1 * PV(soil_swilt_vec, k)) * PV(soil_zse_vec, k) * 1000.0);
    c.csx[0] = c.csx[1] = t.met_ca[0];
    t.met_tvair[0] = t.met_tk[0];
    t.met_qvair[0] = t.met_qv[0];
    t.canopy_tv[0] = t.met_tvair[0];
    t.canopy_fwsoil[0] = 1.0;
    t.canopy_kthlitt[0] = 0.3;
    t.canopy_dvlitt[0] = 3.1415841138194147e-05;
    define_air();
    R qstvair = qsatfjh(t.met_tvair[0] - TFRZ, t.met_pmb[0]);
    t.met_dva[0] = DIV((qstvair - t.met_qvair[0]) * RMAIR, RMH2O) * t.met_pmb[0] * K(100.0);
    c.dsx = t.met_dva[0];
    c.dsx = MAX(c.dsx, K(0.0));
    c.tlfx = t.met_tk[0];
    c.tlfy = t.met_tk[0];
    c.fwsoil = K(1.0);
    // (the plain method's instantiation keeps no such state: stores to these
    // members changed the FP64 kernels' results on gfx950 although nothing
    // reads them, so MODE_PLAIN compiles them out)
    if constexpr (MODE != MODE_PLAIN) vegetated = veg;
    if constexpr (MODE == MODE_HYBRID) {
      // warm start of the leaf fixed point of the first NITER pass at the
      // surrogate's prediction of where that pass converges: leaf
      // temperature, the leaf-surface CO2 of both leaf classes, and the leaf
      // vapour-pressure deficit that temperature implies.  The network is
      // evaluated for sunlit leaf-bearing tiles only; without light (and
      // without predictions) the iteration starts as the reference's does.
      // Those tiles' passes are capped with or without a network, so a run
      // without one is the same capped method from the reference's start
      capped = sunlit_veg;
      if (sunlit_veg && a.pred) {
        c.tlfx = t.met_tk[0] + (R)pred[0];
        c.csx[0] = MAX(K(1.0e-4), t.met_ca[0] * (R)pred[1]);
        c.csx[1] = MAX(K(1.0e-4), t.met_ca[0] * (R)pred[2]);
        c.dsx = MAX(K(0.0), t.met_dva[0] + t.air_dsatdk[0] * (c.tlfx - t.met_tvair[0]));
      }
    }
    R ortsoil = t.ssnow_rtsoil[0];
    int isflag = t.ssnow_isflag[0];
    t.ssnow_tss[0] = (R)(1 - isflag) * t.ssnow_tgg[0] + (R)isflag * t.ssnow_tggsn[0];
    R tss = t.ssnow_tss[0];
    R tss4 = p4(tss);
    t.canopy_fes[0] = 0.;
    t.canopy_fess[0] = 0.;
    t.canopy_fesp[0] = 0.;
    t.ssnow_potev[0] = K(0.);
    t.canopy_fevw_pot[0] = K(0.);
    t.canopy_fhs_cor[0] = K(0.0);
    t.canopy_fns_cor[0] = K(0.0);
    t.canopy_ga_cor[0] = K(0.0);
    radiation(sunlit_veg);
    settled();
    // stability parameter of each NITER pass, kept in registers (zetar(:,1..4));
    // passes 1-3 set zeta1-zeta3 before passes 2-4 read them
    R zeta1 = ZETPOS + K(1), zeta2 = ZETA0, zeta3 = ZETA0;
    t.canopy_zetash[0] = ZETA0;
    t.canopy_zetash[1] = ZETPOS + K(1);
    c.sum_rad_rniso = t.rad_rniso[0] + t.rad_rniso[1];
    c.sum_rad_gradis = t.rad_gradis[0] + t.rad_gradis[1];
    R rt0 = K(0.0), rt1usc = K(0.0);
    int iterplus = 0;
    const R zuv = t.rough_zref_uv[0], ztq = t.rough_zref_tq[0], z0m = t.rough_z0m[0];
    const R disp = t.rough_disp[0], zruffs = t.rough_zruffs[0], z0soilsn = t.rough_z0soilsn[0];
    const R tvrad = t.met_tvrad[0], transd = t.rad_transd[0];
    for (int iter = 1; iter <= 4; iter++) {
      // comp_friction_vel, src/science/canopy/cbl_friction_vel.F90:19-108
      const R zr = iter == 1 ? ZETA0 : iter == 2 ? zeta1 : iter == 3 ? zeta2 : zeta3;
      // the four profile functions take the sign of zr (the heights are
      // positive): one branch, so that their chains of roots, logarithms and
      // exponentials overlap; at zero, in the first pass, they are constants
      // (NaN for an infinite height, as zero times it is).
      // A day of 262,144 tiles in FP64 15.4 -> 15.1 ms, of 4,093 tiles 5.21 ->
      // 5.13 ms, of 1,048,576 in mixed precision 18.1 -> 18.0 ms.
      R mz = MAX(zruffs - disp, z0soilsn);
      R psim_1, psim_2, psis_1, psis_2;
      if (iter == 1) {
        psim_1 = psim_stable(ZETA0) + ZETA0 * zuv;
        psim_2 = psim_stable(ZETA0) + ZETA0 * z0m;
        psis_1 = psis_stable(ZETA0);
        psis_2 = psis_stable(ZETA0) + ZETA0 * mz;
      } else if (stable(zr)) {
        psim_1 = psim_stable(DIV(zr * zuv, ztq));
        psim_2 = psim_stable(DIV(zr * z0m, ztq));
        psis_1 = psis_stable(zr);
        psis_2 = psis_stable(DIV(zr * (mz), ztq));
      } else {
        psim_1 = psim_unstable(DIV(zr * zuv, ztq));
        psim_2 = psim_unstable(DIV(zr * z0m, ztq));
        psis_1 = psis_unstable(zr);
        psis_2 = psis_unstable(DIV(zr * (mz), ztq));
      }
      R rescale = VONK * MAX(t.met_ua[0], UMIN);
      R z_eff = DIV(zuv, z0m);
      R ll = DIV(rescale, log(z_eff) - psim_1 + psim_2);
      t.canopy_us[0] = MIN(MAX(K(1.e-6), ll), K(10.0));
      R us = t.canopy_us[0];
      R xx = K(0.5) + SIGN(K(0.5), ztq + disp - zruffs);
      rt1usc = DIV(xx * (log(DIV(ztq, mz)) - psis_1 + psis_2), VONK);
      const R rt_min = K(5.);
      rt0 = MAX(rt_min, DIV(t.rough_rt0us[0], us));
      t.rough_rt1[0] = MAX(K(5.), DIV(t.rough_rt1usa[0] + t.rough_rt1usb[0] + rt1usc, us));
      R rtsoil = veg ? rt0 : rt0 + t.rough_rt1[0];
      rtsoil = MAX(rt_min, rtsoil);
      if (rtsoil > K(2.) * ortsoil || rtsoil < K(0.5) * ortsoil) rtsoil = MAX(rt_min, K(0.5) * (rtsoil + ortsoil));
      t.ssnow_rtsoil[0] = rtsoil;
      if (veg) {
        R dleaf = PV(veg_dleaf, 0), visc = t.air_visc[0];
        R gbvtop = DIV(DIV(DIV(t.air_cmolar[0] * APOL * visc, PRANDT), dleaf) *
                   sqrt(DIV(DIV(us, MAX(t.rough_usuh[0], K(1.e-6))) * dleaf, visc)) * pow(PRANDT, K(1.0) / K(3.0)),
                   PV(veg_shelrb, 0));
        gbvtop = MAX(K(0.05), gbvtop);
        R coexp = t.rough_coexp[0], extkb = t.rad_extkb[0];
        c.gbhu[0] = DIV(gbvtop * (K(1.0) - exp(-MIN(vlaiw * (K(0.5) * coexp + extkb), K(20.0)))), extkb + K(0.5) * coexp);
        c.gbhu[1] = DIV(K(2.0), coexp) * gbvtop * (K(1.0) - exp(-MIN(K(0.5) * coexp * vlaiw, K(20.0)))) - c.gbhu[0];
      }
      c.rny = c.sum_rad_rniso;
      c.hcy = K(0.0);
      c.ecy = c.rny - c.hcy;
      dryLeaf(c, iter);
      if constexpr (MODE == MODE_CAPTURE) {
        if (iter == 1) {
          tgt[0] = (float)(c.tlfx - t.met_tk[0]);
          tgt[1] = (float)(DIV(c.csx[0], t.met_ca[0]));
          tgt[2] = (float)(DIV(c.csx[1], t.met_ca[0]));
        }
      }
      wetLeaf(c);
      t.canopy_fev[0] = (R)t.canopy_fevc[0] + t.canopy_fevw[0];
      R fwet = t.canopy_fwet[0];
      t.canopy_fhv[0] = (K(1.0) - fwet) * c.hcy + t.canopy_fhvw[0];
      t.canopy_fnv[0] = (K(1.0) - fwet) * c.rny + t.canopy_fevw[0] + t.canopy_fhvw[0];
      if (veg && t.rough_hruff[0] > z0soilsn) {
        t.rad_lwabv[0] = CAPP * RMAIR * (c.tlfy - t.met_tk[0]) * c.sum_rad_gradis;
        R q = DIV(t.rad_lwabv[0], K(2.0) * (K(1.0) - transd) * SBOLTZ * EMLEAF) + p4(tvrad);
        if (q > K(0.0))
          t.canopy_tv[0] = root4(q);
        else
          t.canopy_tv[0] = tvrad;
      } else {
        t.canopy_tv[0] = tvrad;
      }
      t.canopy_fns[0] = t.rad_qssabs[0] + transd * t.met_fld[0] + (K(1.0) - transd) * EMLEAF * SBOLTZ * p4(t.canopy_tv[0]) -
                        EMSOIL * SBOLTZ * tss4;
      t.ssnow_qstss[0] = qsatfjh(tss - TFRZ, t.met_pmb[0]);
      {
        R dq = t.ssnow_qstss[0] - t.met_qv[0];
        R dqu = (R)t.ssnow_rh_srf[0] * t.ssnow_qstss[0] - t.met_qv[0];
        t.ssnow_potev[0] = humidity_deficit_method(dq, dqu);
      }
      latent_heat_flux();
      t.canopy_fhs[0] = DIV(t.air_rho[0] * CAPP * (tss - t.met_tvair[0]), t.ssnow_rtsoil[0]);
      within_canopy(c, rt0, qstvair);
      t.ssnow_qstss[0] = qsatfjh(tss - TFRZ, t.met_pmb[0]);
      {
        R dq = t.ssnow_qstss[0] - t.met_qvair[0];
        R dqu = (R)t.ssnow_rh_srf[0] * t.ssnow_qstss[0] - t.met_qvair[0];
        t.ssnow_potev[0] = humidity_deficit_method(dq, dqu);
      }
      latent_heat_flux();
      t.canopy_fhs[0] = DIV(t.air_rho[0] * CAPP * (tss - t.met_tvair[0]), t.ssnow_rtsoil[0]);
      R fes = (R)t.canopy_fes[0];
      t.canopy_ga[0] = t.canopy_fns[0] - t.canopy_fhs[0] - fes;
      t.canopy_fe[0] = t.canopy_fev[0] + fes;
      t.canopy_fh[0] = t.canopy_fhv[0] + t.canopy_fhs[0];
      if (t.ssnow_potev[0] >= K(0.))
        t.ssnow_potev[0] = MAX(K(0.00001), t.ssnow_potev[0]);
      else
        t.ssnow_potev[0] = MIN(-K(0.0002), t.ssnow_potev[0]);
      if (t.canopy_fevw_pot[0] >= K(0.))
        t.canopy_fevw_pot[0] = MAX(K(0.000001), t.canopy_fevw_pot[0]);
      else
        t.canopy_fevw_pot[0] = MIN(-K(0.002), t.canopy_fevw_pot[0]);
      if constexpr (FULL) {
        t.canopy_rnet[0] = t.canopy_fnv[0] + t.canopy_fns[0];
        t.canopy_rniso[0] = c.sum_rad_rniso + t.rad_qssabs[0] + transd * t.met_fld[0] +
                            (K(1.0) - transd) * EMLEAF * SBOLTZ * p4(tvrad) - EMSOIL * SBOLTZ * p4(tvrad);
        t.canopy_epot[0] = DIV((t.canopy_fevw_pot[0] + DIV(t.ssnow_potev[0], t.ssnow_cls[0])) * dels, t.air_rlam[0]);
        R rll = DIV(t.canopy_epot[0] * t.air_rlam[0], dels);
        if (rll == K(0)) rll = K(1.e-7);
        t.canopy_wetfac_cs[0] = MAX(K(0.), MIN(K(1.0), DIV(t.canopy_fe[0], rll)));
        if (t.canopy_wetfac_cs[0] <= K(0.))
          t.canopy_wetfac_cs[0] =
              MAX(K(0.), MIN(K(1.), MAX(DIV(t.canopy_fev[0], t.canopy_fevw_pot[0]), DIV(fes, t.ssnow_potev[0]))));
      }
      // update_zetar, src/science/canopy/cbl_zetar.F90:13-159
      if (iter < 4) {
        iterplus = (iter + 1 > 2) ? iter + 1 : 2;
        R z = DIV(-(VONK * GRAV * ztq * (t.canopy_fh[0] + K(0.07) * t.canopy_fe[0])),
              t.air_rho[0] * CAPP * t.met_tk[0] * p3(us));
        z = MIN(ZETPOS, z);
        z = MAX(ZETNEG, z);
        if (iterplus == 2) zeta1 = z;
        if (iterplus == 3) zeta2 = z;
        if (iterplus == 4) zeta3 = z;
      }
    }
    t.canopy_zetar[0] = ZETA0;
    t.canopy_zetar[1] = zeta1;
    t.canopy_zetar[2] = zeta2;
    t.canopy_zetar[3] = zeta3;
    if constexpr (MODE == MODE_CAPTURE) {
      // targets 0-2 (above): where the first NITER pass's leaf fixed point
      // settles; 3-7: the step's final leaf temperature, stomatal
      // conductances of both leaf classes, canopy latent and sensible heat
      tgt[3] = (float)(c.tlfx - t.met_tk[0]);
      tgt[4] = (float)t.canopy_gswx[0];
      tgt[5] = (float)t.canopy_gswx[1];
      tgt[6] = (float)c.ecy;
      tgt[7] = (float)c.hcy;
    }
    if constexpr (MODE != MODE_PLAIN) {
      // the previous-step canopy state the next step's surrogate inputs
      // read, written here where it is final rather than held through soil
      // and snow
      if (hyb_out) {
        hyb_out[0] = (float)c.tlfx;
        hyb_out[a.mp] = (float)t.met_tvair[0];
        hyb_out[2 * a.mp] = (float)t.met_qvair[0];
      }
    }
    R us = t.canopy_us[0], ua = t.met_ua[0];
    R rho = t.air_rho[0];
    R rlam = t.air_rlam[0];
    if constexpr (FULL) {
      t.canopy_cduv[0] = DIV(us * us, p2(MAX(ua, UMIN)));
      R lai_min = MAX(LAI_THRESH, vlaiw);
      R rsun = DIV(t.rad_fvlai[0], lai_min), rshd = DIV(t.rad_fvlai[1], lai_min);
      R cc = rsun * t.canopy_gswx[0] + rshd * t.canopy_gswx[1];
      R mincc = MAX(K(1.e-06), cc);
      cc = (K(1.) - transd) * mincc;
      R relm = DIV((R)t.ssnow_wb[0], PV(soil_sfc, 0));
      R sc = transd * p2(K(0.01) * relm);
      R surf = cc + sc;
      if (t.soil_isoilm[0] == ICE_SOIL) surf = K(1.e6);
      t.canopy_gswx_t[0] = surf;
      R z4 = t.canopy_zetar[3];
      t.canopy_cdtq[0] = DIV(t.canopy_cduv[0] * (log(DIV(zuv, z0m)) - psim(DIV(z4 * zuv, ztq)) + psim(DIV(z4 * z0m, ztq))),
                         log(DIV(ztq, K(0.1) * z0m)) - psis(z4) + psis(DIV(z4 * K(0.1) * z0m, ztq)));
      R tstar = DIV(-t.canopy_fh[0], rho * CAPP * us);
      R qstar = DIV(-t.canopy_fe[0], rho * rlam * us * t.ssnow_cls[0]);
      R hruff = t.rough_hruff[0];
      R zscrn = MAX(z0m, K(2.0) - disp);
      R zp = t.canopy_zetar[3];
      (void)iterplus;
      R ftemp = DIV(log(DIV(ztq, zscrn)) - psis(zp) + psis(DIV(zp * zscrn, ztq)), VONK);
      t.canopy_tscrn[0] = t.met_tk[0] - TFRZ - tstar * ftemp;
      R term1 = K(0.), term2 = K(0.), term5 = K(0.), term3 = K(0.), r_sc = K(0.);
      R zscl = MAX(z0soilsn, K(2.0));
      R rghlai = t.canopy_rghlai[0];
      R rt0us = t.rough_rt0us[0], rt1usa = t.rough_rt1usa[0], rt1usb = t.rough_rt1usb[0];
      bool scr = (vlaiw > LAI_THRESH && hruff > K(0.01));
      if (scr) {
        if (disp > K(0.0)) {
          term1 = exp(K(2) * CSW * rghlai * (K(1) - DIV(zscl, hruff)));
          term2 = exp(K(2) * CSW * rghlai * (K(1) - DIV(disp, hruff)));
          term5 = MAX(DIV(K(2.) / K(3.) * hruff, disp), K(1.));
        }
        term3 = A33 * A33 * CTL * K(2) * CSW * rghlai;
        if (zscl < disp) {
          r_sc = DIV(term5 * log(DIV(zscl, z0soilsn)) * (exp(K(2) * CSW * rghlai) - term2), term3);
          r_sc = r_sc + DIV(term5 * log(DIV(disp, zscl)) * (exp(K(2) * CSW * rghlai) - term1), term3);
        } else if (disp <= zscl && zscl < hruff) {
          r_sc = rt0us + DIV(term5 * (term2 - term1), term3);
        } else if (hruff <= zscl && zscl < zruffs) {
          r_sc = rt0us + rt1usa + DIV(term5 * (zscl - hruff), A33 * A33 * CTL * hruff);
        } else if (zscl >= zruffs) {
          r_sc = rt0us + rt1usa + rt1usb +
                 DIV(log(DIV(zscl - disp, MAX(zruffs - disp, z0soilsn))) - psis(DIV((zscl - disp) * zp, ztq)) +
                  psis(DIV((zruffs - disp) * zp, ztq)),
                     VONK);
        }
        t.canopy_tscrn[0] =
            tss + (t.met_tk[0] - tss) * MIN(K(1.), DIV(r_sc, MAX(K(1.), rt0us + rt1usa + rt1usb + rt1usc))) - TFRZ;
      }
      R rsts = qsatfjh(t.canopy_tscrn[0], t.met_pmb[0]);
      R wetfac = t.ssnow_wetfac[0], qv = t.met_qv[0];
      R qtgnet = rsts * wetfac - qv;
      R qsurf = (qtgnet > K(0.)) ? rsts * wetfac : K(0.1) * rsts * wetfac + K(0.9) * qv;
      t.canopy_qmom[0] = rho * (us * us);
      t.canopy_qscrn[0] = qv - qstar * ftemp;
      if (scr)
        t.canopy_qscrn[0] = qsurf + (qv - qsurf) * MIN(K(1.), DIV(r_sc, MAX(K(1.), rt0us + rt1usa + rt1usb + rt1usc)));
    }
    t.canopy_dewmm[0] = DIV(-(MIN(K(0.0), t.canopy_fevw[0]) + (R)MIN(0.0, t.canopy_fevc[0])) * dels, rlam);
    t.canopy_cansto[0] = t.canopy_cansto[0] + t.canopy_dewmm[0];
    t.canopy_cansto[0] = MAX(t.canopy_cansto[0] - DIV(MAX(K(0.0), t.canopy_fevw[0]) * dels, rlam), K(0.0));
    t.canopy_spill[0] = MAX(K(0.0), t.canopy_cansto[0] - c.cansat);
    t.canopy_through[0] = t.canopy_through[0] + t.canopy_spill[0];
    t.canopy_precis[0] = MAX(K(0.), t.canopy_through[0]);
    t.canopy_cansto[0] = t.canopy_cansto[0] - t.canopy_spill[0];
    t.canopy_delwc[0] = t.canopy_cansto[0] - t.canopy_oldcansto[0];
    R tssn = t.ssnow_tss[0];
    t.ssnow_dfn_dtg[0] = DIV((-K(1.)) * K(4.) * EMSOIL * SBOLTZ * tss4, tssn);
    R rttsoil = t.ssnow_rtsoil[0];
    t.ssnow_dfh_dtg[0] = DIV(rho * CAPP, rttsoil);
    t.ssnow_dfe_ddq[0] = DIV(t.ssnow_wetfac[0] * rho * rlam * t.ssnow_cls[0], rttsoil);
    t.ssnow_ddq_dtg[0] = DIV(DIV(RMH2O / RMAIR, t.met_pmb[0]) * TETENA * TETENB * TETENC, p2(TETENC + tssn - TFRZ)) *
                         exp(DIV(TETENB * (tssn - TFRZ), TETENC + tssn - TFRZ));
    t.ssnow_dfe_dtg[0] = t.ssnow_dfe_ddq[0] * t.ssnow_ddq_dtg[0];
    t.canopy_dgdtg[0] = t.ssnow_dfn_dtg[0] - t.ssnow_dfh_dtg[0] - t.ssnow_dfe_dtg[0];
    if constexpr (FULL) {
      R dtl = c.tlfy - t.met_tk[0];
      t.bal_drybal[0] = (c.ecy + c.hcy) - c.sum_rad_rniso + CAPP * RMAIR * dtl * c.sum_rad_gradis;
      t.bal_wetbal[0] = t.canopy_fevw[0] + t.canopy_fhvw[0] - c.sum_rad_rniso * t.canopy_fwet[0] +
                        CAPP * RMAIR * dtl * c.sum_rad_gradis * t.canopy_fwet[0];
      R *qc = t.rad_qcan;
      t.rad_swnet[0] = (qc[0] + qc[1]) + (qc[2] + qc[3]) + t.rad_qssabs[0];
      t.rad_lwnet[0] = t.met_fld[0] - SBOLTZ * EMLEAF * p4(t.canopy_tv[0]) * (K(1) - transd) - t.rad_flws[0] * transd;
      t.rad_rnet[0] = t.rad_swnet[0] + t.rad_lwnet[0];
    }
  }

  // ===================================================================
  // soil and snow; the REAL(r_2) soil water and heat state, its updates and
  // both tridiagonal solves in FP64 (the conductivities' elementary functions
  // in the working precision)

  // src/science/soilsnow/cbl_trimb.F90:17-53
  template <int KMAX>
  CBM_HD static void trimb(const double *a_, const double *b, const double *c, double *rhs) {
    double e[KMAX], temp[KMAX], g[KMAX];
    e[0] = DIV(c[0], b[0]);
#pragma unroll
    for (int k = 1; k < KMAX - 1; k++) {
      temp[k] = DIV(1., b[k] - a_[k] * e[k - 1]);
      e[k] = c[k] * temp[k];
    }
    g[0] = DIV(rhs[0], b[0]);
#pragma unroll
    for (int k = 1; k < KMAX - 1; k++) g[k] = (rhs[k] - a_[k] * g[k - 1]) * temp[k];
    rhs[KMAX - 1] = DIV(rhs[KMAX - 1] - a_[KMAX - 1] * g[KMAX - 2], b[KMAX - 1] - a_[KMAX - 1] * e[KMAX - 2]);
#pragma unroll
    for (int k = KMAX - 2; k >= 0; k--) rhs[k] = g[k] - e[k] * rhs[k + 1];
  }

  // src/science/soilsnow/cbl_snowCheck.F90:9-100
  CBM_HD void snowcheck() {
    R snowd = t.ssnow_snowd[0];
    R *ssdn = t.ssnow_ssdn, *tggsn = t.ssnow_tggsn, *sdepth = t.ssnow_sdepth, *smass = t.ssnow_smass;
    if (snowd <= K(0.0)) {
      t.ssnow_isflag[0] = 0;
      ssdn[0] = ssdn[1] = ssdn[2] = K(120.0);
      t.ssnow_ssdnn[0] = K(120.0);
      tggsn[0] = tggsn[1] = tggsn[2] = TFRZ;
      sdepth[0] = DIV(snowd, ssdn[0]);
      sdepth[1] = K(0.);
      sdepth[2] = K(0.);
      smass[0] = snowd;
      smass[1] = K(0.0);
      smass[2] = K(0.0);
    } else if (snowd < SNMIN * t.ssnow_ssdnn[0]) {
      if (t.ssnow_isflag[0] == 1) {
        ssdn[0] = t.ssnow_ssdnn[0];
        t.ssnow_tgg[0] = tggsn[0];
      }
      t.ssnow_isflag[0] = 0;
      t.ssnow_ssdnn[0] = MIN(K(400.0), MAX(K(120.0), ssdn[0]));
      R tm = MIN(TFRZ, t.ssnow_tgg[0]);
      tggsn[0] = tggsn[1] = tggsn[2] = tm;
      sdepth[0] = DIV(snowd, ssdn[0]);
      sdepth[1] = K(0.0);
      sdepth[2] = K(0.0);
      smass[0] = snowd;
      smass[1] = K(0.0);
      smass[2] = K(0.0);
      ssdn[0] = ssdn[1] = ssdn[2] = t.ssnow_ssdnn[0];
    } else {
      if (t.ssnow_isflag[0] == 0) {
        R tm = MIN(TFRZ, t.ssnow_tgg[0]);
        tggsn[0] = tggsn[1] = tggsn[2] = tm;
        ssdn[1] = ssdn[0];
        ssdn[2] = ssdn[0];
        R tw = t.ssnow_t_snwlr[0];
        sdepth[0] = tw;
        smass[0] = tw * ssdn[0];
        smass[1] = (snowd - smass[0]) * K(0.4);
        smass[2] = (snowd - smass[0]) * K(0.6);
        sdepth[1] = DIV(smass[1], ssdn[1]);
        sdepth[2] = DIV(smass[2], ssdn[2]);
        t.ssnow_ssdnn[0] = DIV(ssdn[0] * smass[0] + ssdn[1] * smass[1] + ssdn[2] * smass[2], snowd);
      }
      t.ssnow_isflag[0] = 1;
    }
  }

  // src/science/soilsnow/cbl_snowDensity.F90:9-102
  CBM_HD void snowdensity() {
    R dels = (R)a.dels;
    R *ssdn = t.ssnow_ssdn, *tggsn = t.ssnow_tggsn, *smass = t.ssnow_smass;
    R snowd = t.ssnow_snowd[0];
    int isflag = t.ssnow_isflag[0];
    R tmin1 = MIN(TFRZ, t.ssnow_tgg[0]);
    if (snowd > K(0.1) && isflag == 0) {
      ssdn[0] = MIN(MAX_SSDN, MAX(K(120.0), ssdn[0] + dels * ssdn[0] * K(3.1e-6) *
                                                     exp(-K(0.03) * (K(273.15) - tmin1) -
                                                         (ssdn[0] >= K(150.0) ? K(0.046) : K(0.0)) * (ssdn[0] - K(150.0)))));
      ssdn[0] = MIN(MAX_SSDN, ssdn[0] + DIV(dels * K(9.806) * ssdn[0] * K(0.75) * snowd,
                                            K(3.0e7) * exp(K(0.021) * ssdn[0] + K(0.081) * (K(273.15) - MIN(TFRZ, t.ssnow_tgg[0])))));
      if (t.soil_isoilm[0] != 9) ssdn[0] = MIN(K(450.0), ssdn[0]);
      t.ssnow_sconds[0] = MAX(K(0.2), MIN(K(2.876e-6) * p2(ssdn[0]) + K(0.074), MAX_SCONDS));
      t.ssnow_sconds[1] = t.ssnow_sconds[0];
      t.ssnow_sconds[2] = t.ssnow_sconds[0];
      t.ssnow_ssdnn[0] = ssdn[0];
      ssdn[1] = ssdn[0];
      ssdn[2] = ssdn[0];
    }
    if (isflag == 1) {
#pragma unroll
      for (int k = 0; k < 3; k++)
        ssdn[k] = ssdn[k] + dels * ssdn[k] * K(3.1e-6) *
                                exp(-K(0.03) * (K(273.15) - MIN(TFRZ, tggsn[k])) -
                                    (ssdn[k] >= K(150.0) ? K(0.046) : K(0.0)) * (ssdn[k] - K(150.0)));
      R tw = t.ssnow_t_snwlr[0];
      ssdn[0] = ssdn[0] + DIV(dels * K(9.806) * ssdn[0] * tw * ssdn[0],
                              K(3.0e7) * exp(K(.021) * ssdn[0] + K(0.081) * (K(273.15) - MIN(TFRZ, tggsn[0]))));
      ssdn[1] = ssdn[1] + DIV(dels * K(9.806) * ssdn[1] * (tw * ssdn[0] + K(0.5) * smass[1]),
                              K(3.0e7) * exp(K(.021) * ssdn[1] + K(0.081) * (K(273.15) - MIN(TFRZ, tggsn[1]))));
      ssdn[2] = ssdn[2] + DIV(dels * K(9.806) * ssdn[2] * (tw * ssdn[0] + smass[1] + K(0.5) * smass[2]),
                              K(3.0e7) * exp(K(.021) * ssdn[2] + K(0.081) * (K(273.15) - MIN(TFRZ, tggsn[2]))));
#pragma unroll
      for (int k = 0; k < 3; k++) t.ssnow_sdepth[k] = DIV(smass[k], ssdn[k]);
      t.ssnow_ssdnn[0] = DIV(ssdn[0] * smass[0] + ssdn[1] * smass[1] + ssdn[2] * smass[2], snowd);
#pragma unroll
      for (int k = 0; k < 3; k++) t.ssnow_sconds[k] = MAX(K(0.2), MIN(K(2.876e-6) * p2(ssdn[k]) + K(0.074), MAX_SCONDS));
    }
  }

  // src/science/soilsnow/cbl_snowAccum.F90:10-188
  CBM_HD void snow_accum() {
    R dels = (R)a.dels;
    R *ssdn = t.ssnow_ssdn, *smass = t.ssnow_smass, *sdepth = t.ssnow_sdepth, *tggsn = t.ssnow_tggsn;
    R psn = t.met_precip_sn[0];
    int isflag = t.ssnow_isflag[0];
    bool notice = t.soil_isoilm[0] != 9;
    R osnowd = t.ssnow_osnowd[0];
    if (t.canopy_precis[0] > K(0.0) && isflag == 0) {
      t.ssnow_snowd[0] = MAX(t.ssnow_snowd[0] + psn, K(0.0));
      t.canopy_precis[0] = t.canopy_precis[0] - psn;
      ssdn[0] = MAX(K(120.0), DIV(ssdn[0] * osnowd, MAX(K(0.01), t.ssnow_snowd[0])) + DIV(K(120.0) * psn, MAX(K(0.01), t.ssnow_snowd[0])));
      t.ssnow_ssdnn[0] = ssdn[0];
      if (t.canopy_precis[0] > K(0.0) && t.ssnow_tgg[0] < TFRZ) {
        R pr = t.canopy_precis[0];
        t.ssnow_snowd[0] = MAX(t.ssnow_snowd[0] + pr, K(0.0));
        R gz = (R)t.ssnow_gammzz[0];
        t.ssnow_tgg[0] = t.ssnow_tgg[0] + DIV(pr * HLF, gz + CSWAT * pr);
        t.ssnow_dtmlt[0] = t.ssnow_dtmlt[0] + DIV(pr * HLF, gz + CSWAT * pr);
        ssdn[0] = MIN(MAX_SSDN, MAX(K(120.0), DIV(ssdn[0] * osnowd, MAX(K(0.01), t.ssnow_snowd[0])) +
                                                  DIV(DENSITY_LIQ * pr, MAX(K(0.01), t.ssnow_snowd[0]))));
        if (notice) ssdn[0] = MIN(K(450.0), ssdn[0]);
        t.canopy_precis[0] = K(0.0);
        t.ssnow_ssdnn[0] = ssdn[0];
      }
    }
    if (t.canopy_precis[0] > K(0.0) && isflag > 0) {
      t.ssnow_snowd[0] = MAX(t.ssnow_snowd[0] + psn, K(0.0));
      t.canopy_precis[0] = t.canopy_precis[0] - psn;
      R osm = smass[0];
      smass[0] = smass[0] + psn;
      ssdn[0] = MAX(K(120.0), DIV(ssdn[0] * osm, smass[0]) + DIV(K(120.0) * psn, smass[0]));
      sdepth[0] = MAX(K(0.02), DIV(smass[0], ssdn[0]));
      if (t.canopy_precis[0] > K(0.0)) {
        R pr = t.canopy_precis[0];
        t.ssnow_snowd[0] = MAX(t.ssnow_snowd[0] + pr, K(0.0));
        R sgamm = ssdn[0] * CGSNOW * sdepth[0];
        osm = smass[0];
        tggsn[0] = tggsn[0] + DIV(pr * HLF * osm, sgamm * osnowd);
        t.ssnow_dtmlt[0] = t.ssnow_dtmlt[0] + DIV(pr * HLF * osm, sgamm * osnowd);
        smass[0] = smass[0] + DIV(pr * osm, osnowd);
        ssdn[0] = MAX(K(120.0), MIN(DIV(ssdn[0] * osm, smass[0]) + DENSITY_LIQ * (K(1.0) - DIV(osm, smass[0])), MAX_SSDN));
        if (notice) ssdn[0] = MIN(K(450.0), ssdn[0]);
        sdepth[0] = DIV(smass[0], ssdn[0]);
#pragma unroll
        for (int k = 1; k < 3; k++) {
          sgamm = ssdn[k] * CGSNOW * sdepth[k];
          osm = smass[k];
          tggsn[k] = tggsn[k] + DIV(pr * HLF * osm, sgamm * osnowd);
          smass[k] = smass[k] + DIV(pr * osm, osnowd);
          ssdn[k] = MAX(K(120.0), MIN(DIV(ssdn[k] * osm, smass[k]) + DENSITY_LIQ * (K(1.0) - DIV(osm, smass[k])), MAX_SSDN));
          if (notice) ssdn[k] = MIN(K(450.0), ssdn[k]);
          sdepth[k] = DIV(smass[k], ssdn[k]);
        }
        t.canopy_precis[0] = K(0.0);
      }
    }
    double fsc = t.canopy_fess[0] + PV(canopy_fes_cor, 0);
    t.canopy_segg[0] = (R)(DIV(fsc, (double)HL));
    t.ssnow_evapsn[0] = K(0);
    if (t.ssnow_cls[0] == K(1.1335)) {
      t.ssnow_evapsn[0] = (R)(DIV((double)dels * fsc, (double)(HL + HLF)));
      R xxx = t.ssnow_evapsn[0];
      isflag = t.ssnow_isflag[0];
      if (isflag == 0 && fsc > 0.0) t.ssnow_evapsn[0] = MIN(t.ssnow_snowd[0], xxx);
      if (isflag > 0 && fsc > 0.0) t.ssnow_evapsn[0] = MIN(K(0.9) * smass[0], xxx);
      t.ssnow_snowd[0] = t.ssnow_snowd[0] - t.ssnow_evapsn[0];
      if (isflag > 0) {
        smass[0] = smass[0] - t.ssnow_evapsn[0];
        sdepth[0] = MAX(K(0.02), DIV(smass[0], ssdn[0]));
      }
      t.canopy_segg[0] = DIV(DIV((HL + HLF) * (xxx - t.ssnow_evapsn[0]), HL), dels);
    }
  }

  // src/science/soilsnow/cbl_snowMelt.F90:9-120
  CBM_HD R snow_melting() {
    R dels = (R)a.dels;
    R snowmlt = K(0.0);
    int isflag = t.ssnow_isflag[0];
    if (t.ssnow_snowd[0] > K(0.0) && isflag == 0 && t.ssnow_tgg[0] >= TFRZ) {
      R gz = (R)t.ssnow_gammzz[0];
      R snowflx = (t.ssnow_tgg[0] - TFRZ) * gz;
      snowmlt = MIN(DIV(snowflx, HLF), t.ssnow_snowd[0]);
      t.ssnow_dtmlt[0] = t.ssnow_dtmlt[0] + DIV(snowmlt * HLF, gz);
      t.ssnow_snowd[0] = t.ssnow_snowd[0] - snowmlt;
      t.ssnow_tgg[0] = t.ssnow_tgg[0] - DIV(snowmlt * HLF, gz);
    }
    if (t.ssnow_snowd[0] > K(0.0) && isflag > 0) {
      R *ssdn = t.ssnow_ssdn, *smass = t.ssnow_smass, *sdepth = t.ssnow_sdepth, *tggsn = t.ssnow_tggsn;
      bool notice = t.soil_isoilm[0] != 9;
      R prev = K(0.0);   // smelt1(k-1) of the reference
      R last = K(0.0);
#pragma unroll
      for (int q = 0; q < 3; q++) {
        R sgamm = ssdn[q] * CGSNOW * sdepth[q];
        R snowflx = DIV(prev * HLF, dels);
        tggsn[q] = tggsn[q] + DIV(snowflx * dels + prev * CSWAT * (TFRZ - tggsn[q]), sgamm + CSWAT * prev);
        R osm = smass[q];
        smass[q] = smass[q] + prev;
        ssdn[q] = MAX(K(120.0), MIN(DIV(ssdn[q] * osm, smass[q]) + DENSITY_LIQ * (K(1.0) - DIV(osm, smass[q])), MAX_SSDN));
        if (notice) ssdn[q] = MIN(K(450.0), ssdn[q]);
        sdepth[q] = DIV(smass[q], ssdn[q]);
        sgamm = smass[q] * CGSNOW;
        R cur = K(0.0);
        if (tggsn[q] > TFRZ) {
          snowflx = (tggsn[q] - TFRZ) * sgamm;
          cur = MIN(DIV(snowflx, HLF), K(0.6) * smass[q]);
          t.ssnow_dtmlt[q] = t.ssnow_dtmlt[q] + DIV(cur * HLF, sgamm);
          smass[q] = smass[q] - cur;
          tggsn[q] = tggsn[q] - DIV(cur * HLF, sgamm);
          sdepth[q] = DIV(smass[q], ssdn[q]);
        }
        prev = cur;
        last = cur;
      }
      // smelt1(:,1) and smelt1(:,2) were zeroed by the next layer's pass
      snowmlt = K(0.0) + K(0.0) + last;
      t.ssnow_snowd[0] = t.ssnow_snowd[0] - snowmlt;
    }
    return snowmlt;
  }

  // src/science/soilsnow/cbl_snowl_adjust.F90:9-156
  CBM_HD void snowl_adjust() {
    if (t.ssnow_isflag[0] <= 0) return;
    R *ssdn = t.ssnow_ssdn, *smass = t.ssnow_smass, *sdepth = t.ssnow_sdepth, *tggsn = t.ssnow_tggsn;
    R tw = t.ssnow_t_snwlr[0], snowd = t.ssnow_snowd[0];
    double excd, excm;
    R osm;
    if (sdepth[0] > tw) {
      excd = (double)sdepth[0] - (double)tw;
      excm = excd * (double)ssdn[0];
      sdepth[0] = sdepth[0] - (R)excd;
      smass[0] = smass[0] - (R)excm;
      osm = smass[1];
      smass[1] = MAX(K(0.01), smass[1] + (R)excm);
      ssdn[1] = (R)MAX(120.0, MIN((double)MAX_SSDN, DIV((double)ssdn[1] * osm, smass[1]) + DIV((double)ssdn[0] * excm, smass[1])));
      sdepth[1] = DIV(smass[1], ssdn[1]);
      tggsn[1] = (R)(DIV((double)tggsn[1] * osm, smass[1]) + DIV((double)tggsn[0] * excm, smass[1]));
      smass[2] = MAX(K(0.01), snowd - smass[0] - smass[1]);
    } else {
      excd = (double)tw - (double)sdepth[0];
      excm = excd * (double)ssdn[1];
      osm = smass[0];
      smass[0] = smass[0] + (R)excm;
      sdepth[0] = tw;
      ssdn[0] = (R)MAX(120.0, MIN((double)MAX_SSDN, DIV((double)ssdn[0] * osm, smass[0]) + DIV((double)ssdn[1] * excm, smass[0])));
      tggsn[0] = (R)(DIV((double)tggsn[0] * osm, smass[0]) + DIV((double)tggsn[1] * excm, smass[0]));
      smass[1] = MAX(K(0.01), smass[1] - (R)excm);
      sdepth[1] = DIV(smass[1], ssdn[1]);
      smass[2] = MAX(K(0.01), snowd - smass[0] - smass[1]);
    }
    double frac = DIV((double)smass[1], MAX(0.02, (double)smass[2]));
    double xfrac = DIV(2.0 / 3.0, frac);
    if (xfrac > 1.0) {
      excm = (xfrac - 1.0) * smass[1];
      osm = smass[1];
      smass[1] = MAX(K(0.01), smass[1] + (R)excm);
      tggsn[1] = DIV(tggsn[1] * osm, smass[1]) + DIV(tggsn[2] * (R)excm, smass[1]);
      ssdn[1] = MAX(K(120.0), MIN(MAX_SSDN, DIV(ssdn[1] * osm, smass[1]) + DIV(ssdn[2] * (R)excm, smass[1])));
      smass[2] = MAX(K(0.01), snowd - smass[0] - smass[1]);
      sdepth[2] = MAX(K(0.02), DIV(smass[2], ssdn[2]));
    } else {
      excm = (1 - xfrac) * smass[1];
      smass[1] = MAX(K(0.01), smass[1] - (R)excm);
      sdepth[1] = MAX(K(0.02), DIV(smass[1], ssdn[1]));
      osm = smass[2];
      smass[2] = MAX(K(0.01), snowd - smass[0] - smass[1]);
      tggsn[2] = DIV(tggsn[2] * osm, smass[2]) + DIV(tggsn[1] * (R)excm, smass[2]);
      ssdn[2] = MAX(K(120.0), MIN(MAX_SSDN, DIV(ssdn[2] * osm, smass[2]) + DIV(ssdn[1] * (R)excm, smass[2])));
      sdepth[2] = DIV(smass[2], ssdn[2]);
    }
    t.ssnow_isflag[0] = 1;
    t.ssnow_ssdnn[0] = DIV(ssdn[0] * sdepth[0] + ssdn[1] * sdepth[1] + ssdn[2] * sdepth[2], sdepth[0] + sdepth[1] + sdepth[2]);
  }

  // src/science/soilsnow/cbl_stempv.F90:13-221 with old_soil_conductivity,
  // src/science/soilsnow/cbl_Oldconductivity.F90:7-59
  CBM_HD void stempv() {
    const double *zse = a.zse;
    double dels = a.dels;
    double at[9], bt[9], ct[9], coeff[10], ccnsw[MS];
#pragma unroll
    for (int r = 0; r < 9; r++) at[r] = 0.0, bt[r] = 1.0, ct[r] = 0.0;
#pragma unroll
    for (int r = 0; r < 10; r++) coeff[r] = 0.0;
    double ssat = PV(soil_ssat, 0);
    bool ice = t.soil_isoilm[0] == 9;
    double cnsd = PV(soil_cnsd, 0);
    const double l60 = log(60.0), l250 = log(250.0);
#pragma unroll
    for (int k = 0; k < MS; k++) {
      if (ice) {
        ccnsw[k] = (double)SNOW_CCNSW;
      } else {
        double ew = (double)(R)(t.ssnow_wblf[k] * ssat);
        double exp_arg = (ew * l60) + (t.ssnow_wbfice[k] * ssat * l250);
        // the conductivity's elementary functions in the working precision
        double f = MAX(1.0, (double)sqrt(MIN(K(2.0), DIV((R)(0.5 * ssat), (R)MIN(ew, 0.5 * ssat)))));
        if (exp_arg > 30)
          ccnsw[k] = 1.5 * f;
        else
          ccnsw[k] = MIN(cnsd * (double)exp((R)exp_arg), 1.5) * f;
      }
    }
    int isflag = t.ssnow_isflag[0];
    double coefa = 0.0, coefb = 0.0;
    double *gammzz = t.ssnow_gammzz;
    double css = PV(soil_css, 0), rhosoil = PV(soil_rhosoil, 0);
    const double dgdtg = t.canopy_dgdtg[0], ga = (double)t.canopy_ga[0];
    if (isflag == 0) {
      double xx = MAX(0., (double)(DIV(t.ssnow_snowd[0], t.ssnow_ssdnn[0])));
      ccnsw[0] = (ccnsw[0] - 0.2) * DIV(zse[0], zse[0] + xx) + 0.2;
#pragma unroll
      for (int k = 3; k <= MS; k++) coeff[k + 2] = DIV(2.0, DIV(zse[k - 2], ccnsw[k - 2]) + DIV(zse[k - 1], ccnsw[k - 1]));
      coeff[4] = DIV(2.0, DIV(zse[0] + xx, ccnsw[0]) + DIV(zse[1], ccnsw[1]));
      coefa = 0.0;
      coefb = coeff[4];
#pragma unroll
      for (int k = 1; k <= MS; k++) {
        double wblfsp = t.ssnow_wblf[k - 1];
        double hcll = (double)t.soil_heat_cap_lower_limit[k - 1];
        gammzz[k - 1] = MAX(hcll, (1.0 - ssat) * css * rhosoil +
                                      ssat * (wblfsp * (double)CSWAT * (double)DENSITY_LIQ +
                                              t.ssnow_wbfice[k - 1] * (double)CSICE * (double)DENSITY_ICE)) *
                        zse[k - 1];
        if (k == 1) gammzz[0] = gammzz[0] + (double)CGSNOW * (double)t.ssnow_snowd[0];
        double dtg = DIV(dels, gammzz[k - 1]);
        at[k + 2] = -dtg * coeff[k + 2];
        ct[k + 2] = -dtg * coeff[k + 3];
        bt[k + 2] = 1.0 - at[k + 2] - ct[k + 2];
      }
      bt[3] = bt[3] - DIV(dgdtg * dels, gammzz[0]);
      t.ssnow_tgg[0] = (R)((double)t.ssnow_tgg[0] + DIV((ga - (double)t.ssnow_tgg[0] * dgdtg) * dels, gammzz[0]));
    } else {
      R *ssdn = t.ssnow_ssdn, *sd = t.ssnow_sdepth, *sc = t.ssnow_sconds;
#pragma unroll
      for (int k = 0; k < 3; k++) sc[k] = MAX(K(0.2), MIN(K(2.876e-6) * p2(ssdn[k]) + K(0.074), MAX_SCONDS));
      coeff[1] = DIV(2.0, (double)(DIV(sd[0], sc[0])) + (double)(DIV(sd[1], sc[1])));
      coeff[2] = DIV(2.0, (double)(DIV(sd[1], sc[1])) + (double)(DIV(sd[2], sc[2])));
      coeff[3] = DIV(2.0, (double)(DIV(sd[2], sc[2])) + DIV(zse[0], ccnsw[0]));
#pragma unroll
      for (int k = 2; k <= MS; k++) coeff[k + 2] = DIV(2.0, DIV(zse[k - 2], ccnsw[k - 2]) + DIV(zse[k - 1], ccnsw[k - 1]));
      coefa = coeff[1];
      coefb = coeff[3];
#pragma unroll
      for (int k = 1; k <= 3; k++) {
        double sgamm = (double)(ssdn[k - 1] * CGSNOW * sd[k - 1]);
        double dtg = DIV(dels, sgamm);
        at[k - 1] = -dtg * coeff[k - 1];
        ct[k - 1] = -dtg * coeff[k];
        bt[k - 1] = 1.0 - at[k - 1] - ct[k - 1];
      }
#pragma unroll
      for (int k = 1; k <= MS; k++) {
        double wblfsp = t.ssnow_wblf[k - 1];
        double hcll = (double)t.soil_heat_cap_lower_limit[k - 1];
        gammzz[k - 1] = MAX((1.0 - ssat) * css * rhosoil +
                                ssat * (wblfsp * (double)CSWAT * (double)DENSITY_LIQ +
                                        t.ssnow_wbfice[k - 1] * (double)CSICE * (double)DENSITY_ICE),
                            hcll) *
                        zse[k - 1];
        double dtg = DIV(dels, gammzz[k - 1]);
        at[k + 2] = -dtg * coeff[k + 2];
        ct[k + 2] = -dtg * coeff[k + 3];
        bt[k + 2] = 1.0 - at[k + 2] - ct[k + 2];
      }
      double sgamm = (double)(ssdn[0] * CGSNOW * sd[0]);
      bt[0] = bt[0] - DIV(dgdtg * dels, sgamm);
      t.ssnow_tggsn[0] = (R)((double)t.ssnow_tggsn[0] + DIV((ga - (double)t.ssnow_tggsn[0] * dgdtg) * dels, sgamm));
    }
    double rhs[9];
#pragma unroll
    for (int k = 0; k < 3; k++) rhs[k] = t.ssnow_tggsn[k];
#pragma unroll
    for (int k = 0; k < MS; k++) rhs[3 + k] = t.ssnow_tgg[k];
    trimb<9>(at, bt, ct, rhs);
#pragma unroll
    for (int k = 0; k < 3; k++) t.ssnow_tggsn[k] = (R)rhs[k];
#pragma unroll
    for (int k = 0; k < MS; k++) t.ssnow_tgg[k] = (R)rhs[3 + k];
    if constexpr (FULL) {
      t.canopy_sghflux[0] = (R)(coefa * (double)(t.ssnow_tggsn[0] - t.ssnow_tggsn[1]));
      t.canopy_ghflux[0] = (R)(coefb * (double)(t.ssnow_tgg[0] - t.ssnow_tgg[1]));
    }
  }

  // src/science/soilsnow/cbl_remove_trans.F90:9-40
  CBM_HD void remove_trans() {
    if (t.canopy_fevc[0] < 0.0) {
      t.canopy_fevw[0] = (R)((double)t.canopy_fevw[0] + t.canopy_fevc[0]);
      t.canopy_fevc[0] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < MS; k++) {
      t.ssnow_wbliq[k] = t.ssnow_wbliq[k] - DIV(t.ssnow_evapfbl[k], PV(soil_zse_vec, k) * 1000.0);
      t.ssnow_wb[k] = t.ssnow_wbliq[k] + t.ssnow_wbice[k];
    }
  }

  // src/science/soilsnow/cbl_soilfreeze.F90:9-81
  CBM_HD void soilfreeze() {
    const double *zse = a.zse;
    const double FL = (double)FROZEN_LIMIT, TF = (double)TFRZ, HF = (double)HLF;
    double ssat = PV(soil_ssat, 0), css = PV(soil_css, 0), rhosoil = PV(soil_rhosoil, 0);
    double base = (double)((R)(K(1.0) - (R)ssat) * (R)css * (R)rhosoil);
#pragma unroll
    for (int k = 0; k < MS; k++) {
      double wb = t.ssnow_wb[k], wbice = t.ssnow_wbice[k], gz = t.ssnow_gammzz[k];
      double tgg = t.ssnow_tgg[k];
      if (tgg < TF && FL * wb - wbice > .001) {
        double sf = MIN(FL * wb - wbice, DIV(ssat - wb, MAX((1.0 - 921.0 / 1000.0), 1.0E-3)));
        sf = MIN(MAX(0.0, sf) * zse[k] * 921.0, DIV((TF - tgg) * gz, HF));
        wbice = MIN(wbice + DIV(sf, zse[k] * 921.0), FL * wb);
        wb = wb + DIV(sf, zse[k] * 921.0) - DIV(sf, zse[k] * 1000.0);
        double a1 = (double)t.soil_heat_cap_lower_limit[k];
        double a2 = base + (wb - wbice) * (4.218e3 * 1000.0) + wbice * (2.100e3 * 921.0);
        gz = MAX(a1, a2) * zse[k];
        if (k == 0 && t.ssnow_isflag[0] == 0) gz = gz + (double)CGSNOW * (double)t.ssnow_snowd[0];
        t.ssnow_tgg[k] = (R)(tgg + DIV(sf * HF, gz));
      } else if (tgg > TF && wbice > 0.) {
        double sm = MIN(wbice * zse[k] * 921.0, DIV((tgg - TF) * gz, HF));
        wbice = MAX(0.0, wbice - DIV(sm, zse[k] * 921.0));
        wb = wb - DIV(sm, zse[k] * 921.0) + DIV(sm, zse[k] * 1000.0);
        double a1 = (double)t.soil_heat_cap_lower_limit[k];
        double a2 = base + (wb - wbice) * (4.218e3 * 1000.0) + wbice * (2.100e3 * 921.0);
        gz = MAX(a1, a2) * zse[k];
        if (k == 0 && t.ssnow_isflag[0] == 0) gz = gz + (double)CGSNOW * (double)t.ssnow_snowd[0];
        t.ssnow_tgg[k] = (R)(tgg - DIV(sm * HF, gz));
      }
      t.ssnow_wb[k] = wb;
      t.ssnow_wbice[k] = wbice;
      t.ssnow_gammzz[k] = gz;
    }
  }

  // src/science/soilsnow/cbl_smoisturev.F90:11-444 (nmeth = -1)
  CBM_HD void smoisturev() {
    const double *zse = a.zse;
    double dels = a.dels;
    double at[MS], bt[MS], ct[MS], fluxh[MS + 1], delt[MS + 1], dtt[MS + 1];
    double *wb = t.ssnow_wb, *wbice = t.ssnow_wbice, *wblf = t.ssnow_wblf;
    double ssat = PV(soil_ssat, 0), hyds = PV(soil_hyds, 0);
    // the power laws of the hydraulic conductivity and diffusivity are
    // evaluated in the working precision; the water state, the fluxes and the
    // tridiagonal system are FP64
    double e1 = (double)PV(soil_i2bp3, 0) - 1;
#pragma unroll
    for (int k = 0; k < MS; k++) at[k] = 0.0, bt[k] = 1.0, ct[k] = 0.0;
    delt[0] = 0.0;
    fluxh[0] = 0.0;
    fluxh[MS] = 0.0;
#pragma unroll
    for (int k = 1; k <= MS - 1; k++) {
      double wbl_k = MAX(0.01, wb[k - 1] - wbice[k - 1]);
      double wbl_kp = MAX(0.01, wb[k] - wbice[k]);
      delt[k] = wbl_kp - wbl_k;
      double wh = MIN(wbl_k, wbl_kp);
      if (wbice[k - 1] > 0.05 || wbice[k] > 0.01) wh = 0.9 * wbl_k + 0.1 * wbl_kp;
      double speed_k = hyds * (double)pow((R)(DIV(wh, ssat)), (R)e1);
      double rat = DIV(delt[k - 1], delt[k] + copysign(1.0e-20, delt[k]));
      double phi = MAX(MAX(0.0, MIN(1.0, 2.0 * rat)), MIN(2.0, rat));
      double fluxhi = wh, fluxlo = wbl_k;
      speed_k = MIN(speed_k, DIV(0.5 * zse[k - 1], dels));
      fluxh[k] = speed_k * (fluxlo + phi * (fluxhi - fluxlo));
    }
    if (wb[MS - 1] > (double)PV(soil_sfc, 0)) {
      double wbl_k = MAX(0.001, wb[MS - 1] - wbice[MS - 1]);
      double wbl_kp = MAX(0.001, ssat - wbice[MS - 1]);
      double wh = MIN(wbl_k, wbl_kp);
      if (wbice[MS - 1] > 0.05) wh = 0.9 * wbl_k + 0.1 * wbl_kp;
      double speed_k = hyds * (double)pow((R)(DIV(wh, ssat)), (R)e1);
      speed_k = DIV(0.5 * speed_k, 1. - MIN(0.5, 10. * wbice[MS - 1]));
      double fluxlo = wbl_k;
      speed_k = MIN(0.5 * speed_k, DIV(0.5 * zse[MS - 1], dels));
      fluxh[MS] = MAX(0.0, speed_k * fluxlo);
    }
#pragma unroll
    for (int k = MS; k >= 1; k--) {
      fluxh[k - 1] = MIN(fluxh[k - 1], DIV((ssat - wb[k - 1]) * zse[k - 1], dels) + fluxh[k]);
      wb[k - 1] = wb[k - 1] + DIV(dels * (fluxh[k - 1] - fluxh[k]), zse[k - 1]);
      double ssatcurr_k = ssat - wbice[k - 1];
      dtt[k] = DIV(dels, zse[k - 1] * ssatcurr_k);
      wblf[k - 1] = DIV(wb[k - 1] - wbice[k - 1], ssatcurr_k);
    }
    t.ssnow_rnof2[0] = (R)(dels * fluxh[MS] * 1000.0);
    double hsbh = PV(soil_hsbh, 0), pwb_min = PV(soil_pwb_min, 0);
    double e2 = (double)PV(soil_ibp2, 0) - 1;
#pragma unroll
    for (int k = 2; k <= MS; k++) {
      double wbh_k = DIV(zse[k - 1] * wblf[k - 2] + zse[k - 2] * wblf[k - 1], zse[k - 1] + zse[k - 2]);
      double fact = (double)pow((R)wbh_k, (R)e2);
      double pwb_wbh =
          (hsbh * (1. - MIN(2. * MIN(0.1, MAX(DIV(wbice[k - 2], MAX(0.01, wb[k - 2])), DIV(wbice[k - 1], MAX(0.01, wb[k - 1])))),
                            0.1))) *
          MAX(pwb_min, wbh_k * fact);
      double z3_k = DIV(pwb_wbh, a.zshh[k - 1]);
      at[k - 1] = -dtt[k] * z3_k;
      ct[k - 2] = -dtt[k - 1] * z3_k;
    }
#pragma unroll
    for (int k = 0; k < MS; k++) bt[k] = 1. - at[k] - ct[k];
    wblf[0] = wblf[0] + DIV(dtt[1] * (double)t.ssnow_fwtop1[0], 1000.0);
    wblf[1] = wblf[1] + DIV(dtt[2] * (double)t.ssnow_fwtop2[0], 1000.0);
    wblf[2] = wblf[2] + DIV(dtt[3] * (double)t.ssnow_fwtop3[0], 1000.0);
    trimb<MS>(at, bt, ct, wblf);
#pragma unroll
    for (int k = 0; k < MS; k++) {
      double ssatcurr = ssat - wbice[k];
      wb[k] = wblf[k] * ssatcurr + wbice[k];
    }
    const double FL = (double)FROZEN_LIMIT;
    double dfactor = (double)(K(1.0) - DENSITY_ICE / DENSITY_LIQ);
#pragma unroll
    for (int k = 0; k < MS; k++) {
      if (wbice[k] > FL * wb[k]) {
        double sicemelt = (double)(R)(DIV(wbice[k] - FL * wb[k], 1.0 - FL * dfactor));
        wbice[k] = wbice[k] - sicemelt;
        wb[k] = wb[k] - dfactor * sicemelt;
        t.ssnow_tgg[k] = (R)((double)t.ssnow_tgg[k] - DIV(sicemelt * zse[k] * 921.0 * (double)HLF, t.ssnow_gammzz[k]));
      }
    }
  }

  // src/science/soilsnow/cbl_surfbv.F90:9-146 (nglacier = 2)
  CBM_HD void surfbv() {
    const double *zse = a.zse;
    R dels = (R)a.dels;
    smoisturev();
    double ssat = PV(soil_ssat, 0);
    double rnof1 = (double)t.ssnow_rnof1[0];
    double wfloor = (double)(DIV(PV(soil_swilt, 0), K(2.) * K(2.0)));
#pragma unroll
    for (int k = 0; k < MS; k++) {
      rnof1 = (double)(R)(rnof1 + (double)(R)(MAX(t.ssnow_wb[k] - ssat, 0.0) * 1000.0) * zse[k]);
      t.ssnow_wb[k] = MAX(wfloor, MIN(t.ssnow_wb[k], ssat));
    }
    t.ssnow_rnof1[0] = (R)rnof1;
    R rnof5 = K(0.);
    R smelt1[4] = {K(0.), K(0.), K(0.), K(0.)};
    R smasstot = K(0.0);
    int isflag = t.ssnow_isflag[0];
    R *smass = t.ssnow_smass;
    if (t.ssnow_snowd[0] > MAX_GLACIER_SNOWD) {
      rnof5 = MIN(K(0.1), t.ssnow_snowd[0] - MAX_GLACIER_SNOWD);
      if (isflag == 0) {
        smasstot = K(0.0);
        t.ssnow_tgg[0] = t.ssnow_tgg[0] - DIV(rnof5 * HLF, (R)(t.ssnow_gammzz[0]));
        t.ssnow_snowd[0] = t.ssnow_snowd[0] - rnof5;
      } else {
        smasstot = smass[0] + smass[1] + smass[2];
      }
    }
#pragma unroll
    for (int k = 1; k <= 3; k++) {
      if (t.ssnow_snowd[0] > MAX_GLACIER_SNOWD && isflag > 0) {
        smelt1[k] = MIN(DIV(rnof5 * smass[k - 1], smasstot), K(0.2) * smass[k - 1]);
        smass[k - 1] = smass[k - 1] - smelt1[k];
        t.ssnow_snowd[0] = t.ssnow_snowd[0] - smelt1[k];
      }
    }
    if (isflag > 0) rnof5 = smelt1[1] + smelt1[2] + smelt1[3];
    t.ssnow_sinfil[0] = K(0.0);
    if (t.veg_iveg[0] == LAKES) {
      R wbl = t.ssnow_wb_lake[0], si;
      R sfc = PV(soil_sfc, 0), swilt = PV(soil_swilt, 0);
      si = MIN(t.ssnow_rnof1[0], wbl);
      t.ssnow_rnof1[0] = MAX(K(0.0), t.ssnow_rnof1[0] - si);
      wbl = MAX(K(0.0), wbl - si);
      si = MIN(t.ssnow_rnof2[0], wbl);
      t.ssnow_rnof2[0] = MAX(K(0.0), t.ssnow_rnof2[0] - si);
      wbl = MAX(K(0.0), wbl - si);
      double z6 = zse[MS - 1];
      double xxx = MAX(0.0, (t.ssnow_wb[MS - 1] - (double)sfc) * z6 * 1000.0);
      si = MIN((R)xxx, wbl);
      t.ssnow_wb[MS - 1] = t.ssnow_wb[MS - 1] - DIV((double)si, z6 * 1000.0);
      wbl = MAX(K(0.0), wbl - si);
      xxx = MAX(0.0, (t.ssnow_wb[MS - 1] - (double)(K(0.5) * (sfc + swilt))) * z6 * 1000.0);
      si = MIN((R)xxx, wbl);
      t.ssnow_wb[MS - 1] = t.ssnow_wb[MS - 1] - DIV((double)si, z6 * 1000.0);
      wbl = MAX(K(0.0), wbl - si);
      t.ssnow_wb_lake[0] = wbl;
      t.ssnow_sinfil[0] = si;
    }
    t.ssnow_rnof1[0] = DIV(t.ssnow_rnof1[0], dels) + DIV(rnof5, dels);
    t.ssnow_rnof2[0] = DIV(t.ssnow_rnof2[0], dels);
    t.ssnow_runoff[0] = t.ssnow_rnof1[0] + t.ssnow_rnof2[0];
  }

  // src/science/soilsnow/cbl_soilsnow_main.F90:28-207
  CBM_HD void soil_snow() {
    const double *zse = a.zse;
    R dels = (R)a.dels;
    if constexpr (FULL) {
      R zsetot = (R)zse[0];
#pragma unroll
      for (int k = 1; k < MS; k++) zsetot = zsetot + (R)zse[k];
      R tg = K(0.);
#pragma unroll
      for (int k = 0; k < MS; k++) tg = tg + (DIV((R)zse[k], zsetot) * t.ssnow_tgg[k]);
      t.ssnow_tggav[0] = tg;
    }
    R css = PV(soil_css, 0), rhosoil = PV(soil_rhosoil, 0), ssat = PV(soil_ssat, 0);
    R hcll = MAX(K(0.01), css * rhosoil);
#pragma unroll
    for (int k = 0; k < MS; k++) t.soil_heat_cap_lower_limit[k] = hcll;
    t.ssnow_t_snwlr[0] = K(0.05);
    t.ssnow_fwtop1[0] = t.ssnow_fwtop2[0] = t.ssnow_fwtop3[0] = K(0.0);
    t.ssnow_runoff[0] = K(0.0);
    t.ssnow_rnof1[0] = K(0.0);
    t.ssnow_rnof2[0] = K(0.0);
    t.ssnow_smelt[0] = K(0.0);
#pragma unroll
    for (int k = 0; k < 3; k++) t.ssnow_dtmlt[k] = K(0.0);
    t.ssnow_osnowd[0] = t.ssnow_snowd[0];
#pragma unroll
    for (int k = 0; k < MS; k++) t.ssnow_wbliq[k] = t.ssnow_wb[k] - t.ssnow_wbice[k];
    if (a.first_call) {
      double xx = (double)(css * rhosoil);
      t.ssnow_gammzz[0] = MAX((double)((K(1.0) - ssat) * css * rhosoil) +
                                  (t.ssnow_wb[0] - t.ssnow_wbice[0]) * (double)CSWAT * (double)DENSITY_LIQ +
                                  t.ssnow_wbice[0] * (double)CSICE * (double)DENSITY_ICE,
                              xx) * zse[0] +
                          (double)((K(1.) - (R)t.ssnow_isflag[0]) * CGSNOW * t.ssnow_snowd[0]);
    }
#pragma unroll
    for (int k = 0; k < MS; k++) {
      t.ssnow_wblf[k] = DIV(MAX(0.01, (t.ssnow_wb[k] - t.ssnow_wbice[k])), (double)ssat);
      t.ssnow_wbfice[k] = (double)(R)(DIV(t.ssnow_wbice[k], (double)ssat));
    }
    snowcheck();
    snowdensity();
    snow_accum();
    R snowmlt = snow_melting();
    t.ssnow_smelt[0] = snowmlt;
    snowl_adjust();
    stempv();
    int isflag = t.ssnow_isflag[0];
    t.ssnow_tss[0] = (R)(1 - isflag) * t.ssnow_tgg[0] + (R)isflag * t.ssnow_tggsn[0];
    snowmlt = snow_melting();
    t.ssnow_smelt[0] = t.ssnow_smelt[0] + snowmlt;
    remove_trans();
    soilfreeze();
    R totwet = t.canopy_precis[0] + t.ssnow_smelt[0];
    double weting = (double)totwet + MAX(0.0, (double)t.ssnow_pudsto[0] - DIV(t.canopy_fesp[0], (double)HL) * (double)dels);
    double dssat = (double)ssat;
    double xxx = dssat - t.ssnow_wb[0];
    double sinfil1 = MIN(0.95 * xxx * zse[0] * 1000.0, weting);
    xxx = dssat - t.ssnow_wb[1];
    double sinfil2 = MIN(0.95 * xxx * zse[1] * 1000.0, weting - sinfil1);
    xxx = dssat - t.ssnow_wb[2];
    double sinfil3 = MIN(0.95 * xxx * zse[2] * 1000.0, weting - sinfil1 - sinfil2);
    t.ssnow_fwtop1[0] = (R)(DIV(sinfil1, (double)dels) - (double)t.canopy_segg[0]);
    t.ssnow_fwtop2[0] = (R)(DIV(sinfil2, (double)dels));
    t.ssnow_fwtop3[0] = (R)(DIV(sinfil3, (double)dels));
    R pudsto = (R)MAX(0.0, weting - sinfil1 - sinfil2 - sinfil3);
    t.ssnow_rnof1[0] = MAX(K(0.), pudsto - (R)PV(ssnow_pudsmx, 0));
    t.ssnow_pudsto[0] = pudsto - t.ssnow_rnof1[0];
    surfbv();
    t.ssnow_smelt[0] = DIV(t.ssnow_smelt[0], dels);
    isflag = t.ssnow_isflag[0];
    t.ssnow_tss[0] = (R)(1 - isflag) * t.ssnow_tgg[0] + (R)isflag * t.ssnow_tggsn[0];
#pragma unroll
    for (int k = 0; k < MS; k++) t.ssnow_wbliq[k] = t.ssnow_wb[k] - t.ssnow_wbice[k];
    if constexpr (FULL) t.ssnow_totsdepth[0] = t.ssnow_sdepth[0] + t.ssnow_sdepth[1] + t.ssnow_sdepth[2];
    double wbtot = 0.0;
#pragma unroll
    for (int k = 0; k < MS; k++) wbtot = wbtot + (t.ssnow_wbliq[k] * 1000.0 + t.ssnow_wbice[k] * 921.0) * zse[k];
    t.ssnow_wbtot[0] = wbtot;
  }

  // src/science/soilsnow/cbl_snow_aging.F90:11-83
  CBM_HD void snow_aging() {
    R snowd = t.ssnow_snowd[0];
    if (snowd > K(1.0)) {
      R dnsnow = MIN(K(1.0), K(0.1) * MAX(K(0.0), snowd - t.ssnow_osnowd[0]));
      int fl = t.ssnow_isflag[0];
      R tmp = (R)fl * t.ssnow_tggsn[0] + (R)(1 - fl) * t.ssnow_tgg[0];
      tmp = MIN(tmp, TFRZ);
      R ar1 = K(5000.0) * (K(1.0) / (TFRZ - K(0.01)) - DIV(K(1.0), tmp));
      R ar2 = K(10.0) * ar1;
      R ar3;
      if (t.soil_isoilm[0] == 9) {
        ar3 = K(0.0000001);
        dnsnow = K(1.0);
      } else {
        ar3 = K(0.1);
      }
      R dtau = K(1.0e-6) * (exp(ar1) + exp(ar2) + ar3) * (R)a.dels;
      t.ssnow_snage[0] = MAX(K(0.0), (t.ssnow_snage[0] + dtau) * (K(1.0) - dnsnow));
    }
  }

  // src/science/misc/cable_carbon.F90:38-360 (mvtype 17, DIAG_SOIL_RESP on)
  CBM_HD static R rw17(int i) {
    const R v[17] = {K(16.), K(16.), K(18.), K(8.7), K(12.5), K(15.1), K(10.4), K(7.5), K(6.1),
                     K(6.1), K(0.001), K(5.8), K(0.001), K(5.8), K(0.001), K(9.0), K(0.001)};
    return v[i];
  }
  CBM_HD static R tfcl17(int i) {
    const R v[17] = {K(0.42), K(0.248), K(0.38), K(0.345), K(0.31), K(0.73), K(2.4), K(0.35), K(0.997),
                     K(0.997), K(0.9500), K(0.55), K(0.9500), K(0.55), K(0.9500), K(2.4), K(0.9500)};
    return v[i];
  }
  CBM_HD static R tvclst17(int i) {
    const R v[17] = {K(235.), K(283.), K(268.), K(278.), K(278.), K(235.), K(278.0), K(278.0),
                     K(278.0), K(278.0), K(278.0), K(278.), K(278.), K(278.), K(268.), K(278.), K(278.)};
    return v[i];
  }
  CBM_HD void carbon() {
    R dels = (R)a.dels;
    R rc0 = (R)a.ratecp[0], rc1 = (R)a.ratecp[1], rc2 = (R)a.ratecp[2];
    R *cp = t.bgc_cplant, *cs = t.bgc_csoil;
    R S = rc0 * cp[0] + rc1 * cp[1] + rc2 * cp[2];
    R pc1 = (S - rc0 * cp[0]);
    R pc1w = (S - rc0 * cp[0] - rc2 * cp[2]);
    R pc1r = (S - rc0 * cp[0] - rc1 * cp[1]);
    R tk = t.met_tk[0];
    R tmp1 = MAX(K(3.22) - K(0.046) * (tk - TFRZ), K(1e-6));
    R tmp2 = K(0.1) * (tk - TFRZ - K(20.0));
    R tmp3 = pow(tmp1, tmp2);
    const R spy = K(365.0) * K(24.0) * K(3600.0);
    R rp20 = PV(veg_rp20, 0);
    R frp = DIV(rp20 * tmp3 * pc1, spy);
    R frpw = DIV(rp20 * tmp3 * pc1w, spy);
    R frpr = DIV(rp20 * tmp3 * pc1r, spy);
    t.canopy_frp[0] = frp;
    t.canopy_frpw[0] = frpw;
    t.canopy_frpr[0] = frpr;
    R swilt = PV(soil_swilt, 0);
    {
      const R t0 = K(-46.0), rswch = K(0.16), soilcf = K(1.0);
      R den = MAX(K(0.07), PV(soil_sfc, 0) - swilt);
      R rswc = DIV(MAX(K(0.0001), PV(veg_froot, 0) * ((R)t.ssnow_wb[1] - swilt)), den);
      R tsoil = PV(veg_froot, 0) * t.ssnow_tgg[1] - TFRZ;
      R tref = MAX(K(0.), t.ssnow_tgg[MS - 1] - (TFRZ - K(.05)));
#pragma unroll
      for (int k = 1; k < MS; k++) {
        rswc = rswc + DIV(MAX(K(0.0001), PV(veg_froot, k) * ((R)t.ssnow_wb[k] - swilt)), den);
        tsoil = tsoil + PV(veg_froot, k) * t.ssnow_tgg[k];
      }
      rswc = MIN(K(1.), rswc);
      tsoil = MAX(t0 + K(2.), tsoil);
      R e0rswc = K(52.4) + K(285.) * rswc;
      R ftsoil = MIN(K(0.0015), DIV(K(1.), tref - t0) - DIV(K(1.), tsoil - t0));
      R sss = MAX(K(-15.), MIN(K(1.), e0rswc * ftsoil));
      R ftsrs = exp(sss);
      t.canopy_frs[0] = DIV(PV(veg_vegcf, 0) * (K(144.0) / K(44.0e6)) * soilcf * MIN(K(1.), K(1.4) * MAX(K(.3), K(.0278) * tsoil + K(.5))) *
                        ftsrs * rswc, rswch + rswc);
    }
    {
      const R beta = K(0.9), trnl = K(3.17e-8), trnr = K(4.53e-9), trnsf = K(1.057e-10), trnw = K(6.342e-10);
      int iv = t.veg_iveg[0] - 1;
      R coef_cold = exp(MIN(K(1.), -(t.canopy_tv[0] - tvclst17(iv))));
      R wbav = PV(veg_froot, 0) * (R)t.ssnow_wb[0];
#pragma unroll
      for (int k = 1; k < MS; k++) wbav = wbav + PV(veg_froot, k) * (R)t.ssnow_wb[k];
      wbav = MAX(K(0.01), wbav);
      R ce = K(2.0) - PV(soil_ibp2, 0);
      R esw = pow(wbav, ce) - K(1.0);
      esw = MAX(K(1.0), esw);
      R eswilt = pow(swilt, ce) - K(1.0);
      R rel = DIV(esw, eswilt) - K(1.0);
      rel = MIN(K(1.0), rel);
      R coef_drght = exp(K(5.0) * rel);
      R coef_cd = (coef_cold + coef_drght) * K(2.0e-7);
      R fcl = exp(-tfcl17(iv) * t.veg_vlai[0]);
      R clitt = (coef_cd + trnl) * cp[0];
      R fpn = t.canopy_fpn[0];
      cp[0] = cp[0] - dels * (fpn * fcl + clitt);
      R fr = MIN(K(1.), DIV(exp(DIV(-rw17(iv) * beta * K(0.0001) * cp[2], MAX(cp[1], K(0.01)))), beta));
      R cfwd = trnw * cp[1];
      cp[1] = cp[1] - dels * (fpn * (K(1.) - fcl) * (K(1.) - fr) + frpw + cfwd);
      R cfrts = trnr * cp[2];
      cp[2] = cp[2] - dels * (fpn * (K(1.) - fcl) * fr + cfrts + frpr);
      R cfsf = trnsf * cs[0];
      R frs = t.canopy_frs[0];
      cs[0] = cs[0] + dels * (K(0.98) * clitt + K(0.9) * cfrts + cfwd - cfsf - K(0.98) * frs);
      cs[1] = cs[1] + dels * (K(0.02) * clitt + K(0.1) * cfrts + cfsf - K(0.02) * frs);
#pragma unroll
      for (int k = 0; k < 3; k++) cp[k] = MAX(K(0.00), cp[k]);
#pragma unroll
      for (int k = 0; k < 2; k++) cs[k] = MAX(K(0.00), cs[k]);
    }
  }

  // ===================================================================
  // src/offline/cbl_model_driver_offline.F90:38-231, with the offline
  // driver's contract (src/offline/cable_serial.F90:572-575, 602-605,
  // 725-729) and the balance accumulators (src/offline/cable_checks.F90
  // :472-618) in FP64
  CBM_HD void run() {
    run([] {}, [] {}, [] {}, [] {});
  }
  // `late` runs after the canopy and before soil and snow: the resident
  // kernel takes there, from LDS, the state that only soil, snow, carbon and
  // the balances read, so it is not held in registers through the canopy
  // iteration (the drop-in kernel loads it there).  `tail` runs after soil and
  // snow, before the flux totals and carbon: the resident kernel takes there
  // the driver's running sums, which sumcflux reads after the step.
  // `stash` runs before the canopy, `settled` in it before the leaf iteration,
  // when the radiation, roughness and air diagnostics have their last values.
  template <class Late, class Tail, class Stash, class Settled>
  CBM_HD void run(Late &&late, Tail &&tail, Stash &&stash, Settled &&settled) {
    R dels = (R)a.dels;
    if (a.driver) {
      // the offline driver before cbm, src/offline/cable_serial.F90:572-575
      t.met_ofsd[0] = t.met_fsd[0] + t.met_fsd[1];
      t.canopy_oldcansto[0] = t.canopy_cansto[0];
      if (t.veg_iveg[0] >= 14) t.veg_vlai[0] = K(0.);
    }
    if (t.veg_iveg[0] == LAKES && t.ssnow_wb[0] < (double)PV(soil_sfc, 0)) {
      t.ssnow_wbtot1[0] = (R)((t.ssnow_wb[0]) * 1000.0 * a.zse[0]);
      t.ssnow_wb[0] = (double)PV(soil_sfc, 0);
      t.ssnow_wbtot2[0] = (R)((t.ssnow_wb[0]) * 1000.0 * a.zse[0]);
    }
    t.ssnow_wb_lake[0] = t.ssnow_wb_lake[0] + MAX(t.ssnow_wbtot2[0] - t.ssnow_wbtot1[0], K(0.));
    ruff_resist();
    define_air();
    bool veg_mask = t.canopy_vlaiw[0] > LAI_THRESH;
    bool sunlit = (t.met_fsd[0] + t.met_fsd[1]) > RAD_THRESH;
    bool sunlit_veg = veg_mask && sunlit;
    init_radiation_albedo(veg_mask);
    t.rad_albedo_t[0] = (t.rad_albedo[0] + t.rad_albedo[1]) * K(0.5);
    t.ssnow_otss_0[0] = t.ssnow_otss[0];
    t.ssnow_otss[0] = t.ssnow_tss[0];
    stash();
    define_canopy(sunlit_veg, settled);
    late();
    t.ssnow_owetfac[0] = t.ssnow_wetfac[0];
    soil_snow();
    snow_aging();
    tail();
    t.ssnow_deltss[0] = t.ssnow_tss[0] - t.ssnow_otss[0];
    t.canopy_fev[0] = (R)t.canopy_fevc[0] + t.canopy_fevw[0];
    t.canopy_fe[0] = (R)((double)t.canopy_fev[0] + t.canopy_fes[0]);
    t.canopy_rnet[0] = t.canopy_fns[0] + t.canopy_fnv[0];
    R transd = t.rad_transd[0];
    t.rad_trad[0] = root4((K(1.) - transd) * p4(t.canopy_tv[0]) + transd * p4(t.ssnow_tss[0]));
    carbon();
    R fpn = t.canopy_fpn[0];
    t.canopy_fnpp[0] = -K(1.0) * fpn - t.canopy_frp[0];
    t.canopy_fgpp[0] = -K(1.0) * fpn + t.canopy_frday[0];
    t.canopy_fnee[0] = fpn + t.canopy_frs[0] + t.canopy_frp[0];
    t.canopy_fra[0] = t.canopy_frp[0] + t.canopy_frday[0];
    if (!a.driver) return;
    // the offline driver after cbm: unit conversions,
    // src/offline/cable_serial.F90:602-605, then the balance checks
    t.ssnow_smelt[0] = t.ssnow_smelt[0] * dels;
    t.ssnow_rnof1[0] = t.ssnow_rnof1[0] * dels;
    t.ssnow_rnof2[0] = t.ssnow_rnof2[0] * dels;
    t.ssnow_runoff[0] = t.ssnow_runoff[0] * dels;
    // mass_balance, src/offline/cable_checks.F90:472-551 (FP64 accumulators,
    // evaluated exactly as written in every build of this file)
    {
#pragma float_control(precise, on)
      if (a.ktau == 1) t.drv_owb[0] = t.ssnow_wbtot[0];
      double delwb = t.ssnow_wbtot[0] - t.drv_owb[0];
      t.drv_owb[0] = t.ssnow_wbtot[0];
      double rlam = (double)t.air_rlam[0], cls = (double)t.ssnow_cls[0], dd = (double)dels;
      double wbal = (double)t.met_precip[0] - (double)t.canopy_delwc[0] - (double)t.ssnow_snowd[0] +
                    (double)t.ssnow_osnowd[0] - (double)t.ssnow_runoff[0] -
                    ((double)t.canopy_fevw[0] + t.canopy_fevc[0] + t.canopy_fes[0] / cls) * dd / rlam - delwb -
                    PV(ssnow_qrecharge, 0);
      t.bal_wbal[0] = (R)wbal;
      if (a.ktau == 1) {
        t.bal_wbal_tot[0] = 0.;
        t.bal_precip_tot[0] = 0.;
        t.bal_rnoff_tot[0] = 0.;
        t.bal_evap_tot[0] = 0.;
      }
      if (a.ktau > 10) {
        t.bal_wbal_tot[0] = t.bal_wbal_tot[0] + (double)t.bal_wbal[0];
        t.bal_precip_tot[0] = t.bal_precip_tot[0] + (double)t.met_precip[0];
        t.bal_rnoff_tot[0] = t.bal_rnoff_tot[0] + (double)t.ssnow_rnof1[0] + (double)t.ssnow_rnof2[0];
        t.bal_evap_tot[0] = t.bal_evap_tot[0] + ((double)t.canopy_fev[0] + t.canopy_fes[0] / cls) * dd / rlam;
      }
    }
    // energy_balance, src/offline/cable_checks.F90:565-618
    {
#pragma float_control(precise, on)
      R *fsd = t.met_fsd, *alb = t.rad_albedo, *qc = t.rad_qcan;
      R tv4 = p4(t.canopy_tv[0]);
      R radbal = fsd[0] + fsd[1] + t.met_fld[0] - alb[0] * fsd[0] - alb[1] * fsd[1] -
                 (EMSOIL * SBOLTZ * transd * p4(t.ssnow_otss[0])) - (EMLEAF * SBOLTZ * (K(1) - transd) * tv4) -
                 t.canopy_fnv[0] - t.canopy_fns[0];
      R fes = (R)t.canopy_fes[0];
      R ebal = (qc[0] + qc[1]) + (qc[2] + qc[3]) + t.rad_qssabs[0] + t.met_fld[0] - SBOLTZ * EMLEAF * tv4 * (K(1) - transd) -
               t.rad_flws[0] * transd - t.canopy_fev[0] - fes - t.canopy_fh[0] - t.canopy_ga[0];
      t.bal_radbal[0] = radbal;
      t.bal_ebal[0] = ebal;
      if constexpr (FULL) {
        t.bal_ebalsoil[0] = t.canopy_fns[0] - fes - t.canopy_fhs[0] - t.canopy_ga[0];
        t.bal_ebalveg[0] = t.canopy_fnv[0] - t.canopy_fev[0] - t.canopy_fhv[0];
      }
      t.bal_ebal_tot[0] = t.bal_ebal_tot[0] + (double)ebal;
      t.bal_radbalsum[0] = t.bal_radbalsum[0] + (double)radbal;
    }
  }

  // the offline driver's running carbon sums after the step (driver mode):
  // sumcflux, src/offline/casa_cable.F90:482-560 with icycle = 0 and
  // kstart = 1, called at src/offline/cable_serial.F90:713-715.  The fnee it
  // sets is cbm's own (run above).  The caller has the previous step's sums
  // in t (the resident run loads them in run's `tail`).
  CBM_HD void sumcflux() {
    const R dels = (R)a.dels;
    const R pn = t.canopy_fpn[0] * dels, rd = t.canopy_frday[0] * dels;
    const R rpw = t.canopy_frpw[0] * dels, rpr = t.canopy_frpr[0] * dels;
    const R rp = t.canopy_frp[0] * dels, rs = t.canopy_frs[0] * dels;
    if (a.ktau == 1) {
      t.sum_flux_sumpn[0] = pn;
      t.sum_flux_sumrd[0] = rd;
      t.sum_flux_dsumpn[0] = pn;
      t.sum_flux_dsumrd[0] = rd;
      t.sum_flux_sumrpw[0] = rpw;
      t.sum_flux_sumrpr[0] = rpr;
      t.sum_flux_sumrp[0] = rp;
      t.sum_flux_dsumrp[0] = rp;
      t.sum_flux_sumrs[0] = rs;
    } else {
      t.sum_flux_sumpn[0] = t.sum_flux_sumpn[0] + pn;
      t.sum_flux_sumrd[0] = t.sum_flux_sumrd[0] + rd;
      t.sum_flux_dsumpn[0] = t.sum_flux_dsumpn[0] + pn;
      t.sum_flux_dsumrd[0] = t.sum_flux_dsumrd[0] + rd;
      t.sum_flux_sumrpw[0] = t.sum_flux_sumrpw[0] + rpw;
      t.sum_flux_sumrpr[0] = t.sum_flux_sumrpr[0] + rpr;
      t.sum_flux_sumrp[0] = t.sum_flux_sumrp[0] + rp;
      t.sum_flux_dsumrp[0] = t.sum_flux_dsumrp[0] + rp;
      t.sum_flux_sumrs[0] = t.sum_flux_sumrs[0] + rs;
    }
  }
};

}  // namespace cbm
