// host_resident.hip -- the resident step as the GPU runs it, compiled for the
// CPU: run_tile of cable_amd/csrc/cbm_kernel.h, several steps of a tile with
// the late state in a lane's slots, class tables in the step's precision and
// derived columns, beside the drop-in step on the same inputs
// (tests/test_host_resident.py builds and drives it).
//
//   host_resident IN OUT
//
// IN (little-endian): int64 mp, int32 nsteps, int32 precision (0 FP64, 1
// mixed), double dels, 18 doubles zse(6) zshh(7) ratecp(3) ratecs(2), the veg
// and soil class tables (17 x cable_gpu_veg_cols, 9 x cable_gpu_soil_cols
// doubles), every field of include/cable_fields.h in table order as (n, mp)
// doubles, then per step the forcing fields in table order.  OUT: every field
// after the last step, as doubles: by the drop-in steps, then by run_tile.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "../cable_amd/csrc/cbm_kernel.h"

using namespace cbm;

namespace {
struct Meta {
  char prec;
  int n, role;
};
const Meta META[] = {
#define PARAM ROLE_PARAM
#define FORC ROLE_FORC
#define STATE ROLE_STATE
#define DIAG ROLE_DIAG
#define X(id, name, prec, n, role) {#prec[0], n, role},
    CABLE_FIELDS(X)
#undef X
#undef PARAM
#undef FORC
#undef STATE
#undef DIAG
};
// the resident run's forcing
const int COMPACT[] = {CABLE_F_met_fsd, CABLE_F_met_fld, CABLE_F_met_tk,     CABLE_F_met_qv,
                       CABLE_F_met_ua,  CABLE_F_met_pmb, CABLE_F_met_precip, CABLE_F_met_coszen};

bool rd(FILE *f, void *p, size_t n) { return fread(p, 1, n, f) == n; }

// an array in the device type of field i, left unset
template <class R>
struct Field {
  int kind;  // 0 double, 1 float, 2 int
  void *p;
  Field(int i, size_t n) {
    const char c = META[i].prec;
    kind = c == 'I' ? 2 : c == 'D' || c == 'B' || sizeof(R) == 8 ? 0 : 1;
    p = malloc(n * (kind == 0 ? 8 : 4));
  }
  void put(size_t j, double v) {
    if (kind == 0) ((double *)p)[j] = v;
    else if (kind == 1) ((float *)p)[j] = (float)v;
    else ((int *)p)[j] = (int)v;
  }
  double get(size_t j) const { return kind == 0 ? ((double *)p)[j] : kind == 1 ? ((float *)p)[j] : ((int *)p)[j]; }
};

template <class R>
int run(FILE *in, FILE *out, int64_t mp, int nsteps, double dels, const double *glob, const std::vector<double> &vtab,
        const std::vector<double> &stab) {
  std::vector<Field<R>> full, res;
  std::vector<void *> F(CABLE_NFIELDS), G(CABLE_NFIELDS);
  std::vector<double> h;
  for (int i = 0; i < CABLE_NFIELDS; i++) {
    const size_t n = (size_t)META[i].n * mp;
    h.resize(n);
    if (!rd(in, h.data(), sizeof(double) * n)) return 2;
    full.emplace_back(i, n);
    res.emplace_back(i, n);
    for (size_t j = 0; j < n; j++) {
      full[i].put(j, h[j]);
      res[i].put(j, h[j]);
    }
    F[i] = full[i].p;
    G[i] = res[i].p;
  }
  std::vector<Field<R>> met;
  for (int i : COMPACT) {
    met.emplace_back(i, (size_t)nsteps * mp);
    G[i] = met.back().p;
  }
  StepArgs a;
  memset(&a, 0, sizeof a);
  a.mp = mp;
  a.driver = 1;
  a.dels = dels;
  memcpy(a.zse, glob, sizeof a.zse);
  memcpy(a.zshh, glob + 6, sizeof a.zshh);
  memcpy(a.ratecp, glob + 13, sizeof a.ratecp);
  memcpy(a.ratecs, glob + 16, sizeof a.ratecs);
  std::vector<StepArgs> args;
  for (int s = 0; s < nsteps; s++) {
    for (int i = 0; i < CABLE_NFIELDS; i++) {
      if (META[i].role != ROLE_FORC) continue;
      const size_t n = (size_t)META[i].n * mp;
      h.resize(n);
      if (!rd(in, h.data(), sizeof(double) * n)) return 2;
      for (size_t j = 0; j < n; j++) full[i].put(j, h[j]);
      for (size_t q = 0; q < met.size(); q++)
        if (COMPACT[q] == i)
          for (int64_t j = 0; j < mp; j++) met[q].put((size_t)s * mp + j, h[j]);
      if (i == CABLE_F_met_ca) a.ca = h[0];
      if (i == CABLE_F_met_doy) a.doy = h[0];
    }
    a.ktau = s + 1;
    a.first_call = s == 0;
    a.F = F.data();
    a.foff = 0;
    for (int64_t t = 0; t < mp; t++) {
      TileOut<MODE_PLAIN, false> o;
      step_tile<R, true, false, MODE_PLAIN, false>(a, t, nullptr, nullptr, o);
    }
    a.F = G.data();
    a.foff = (int64_t)s * mp;
    args.push_back(a);
  }
  // the class tables as a workgroup stages them
  std::vector<R> lv(vtab.size()), ls(stab.size()), lx(NVEGCLASS * VX_N);
  std::vector<double> lvd(sizeof(R) == 4 ? NVEGCLASS * NVEGD : 0), lsd(sizeof(R) == 4 ? stab.size() : 0);
  for (size_t i = 0; i < vtab.size(); i++) put_veg((int)i, vtab[i], lv.data(), lvd.data());
  for (size_t i = 0; i < stab.size(); i++) put_soil((int)i, stab[i], ls.data(), lsd.data());
  for (size_t i = 0; i < lx.size(); i++) lx[i] = derived_column<R>((int)i, lv.data());
  using Late = LateStage<R>;
  for (int64_t t = 0; t < mp; t++) {
    // a lane's slots in buffers that end with its last one, unset
    const int lane = (int)(t % Late::LANES);
    Late late;
    auto *f = (decltype(late.f))malloc(sizeof *late.f * ((Late::NF - 1) * Late::LANES + lane + 1));
    auto *d = (double *)malloc(sizeof(double) * ((Late::ND - 1) * Late::LANES + lane + 1));
    late.f = f + lane;
    late.d = d + lane;
    run_tile<R>(args.data(), nsteps, t, true, lv.data(), ls.data(), late, lx.data(), lvd.data(), lsd.data());
    free(f);
    free(d);
  }
  for (auto *set : {&full, &res})
    for (int i = 0; i < CABLE_NFIELDS; i++) {
      h.resize((size_t)META[i].n * mp);
      for (size_t j = 0; j < h.size(); j++) h[j] = (*set)[i].get(j);
      if (fwrite(h.data(), sizeof(double), h.size(), out) != h.size()) return 3;
    }
  for (auto *set : {&full, &res, &met})
    for (auto &x : *set) free(x.p);
  return 0;
}
}  // namespace

int main(int argc, char **argv) {
  if (argc != 3) {
    fprintf(stderr, "usage: host_resident IN OUT\n");
    return 1;
  }
  FILE *in = fopen(argv[1], "rb"), *out = fopen(argv[2], "wb");
  if (!in || !out) return 1;
  int64_t mp = 0;
  int32_t nsteps = 0, precision = 0;
  double dels = 0, glob[18];
  if (!rd(in, &mp, 8) || !rd(in, &nsteps, 4) || !rd(in, &precision, 4) || !rd(in, &dels, 8) ||
      !rd(in, glob, sizeof glob))
    return 2;
  std::vector<double> vtab(NVEGCLASS * VC_N), stab(NSOILCLASS * SC_N);
  if (!rd(in, vtab.data(), sizeof(double) * vtab.size()) || !rd(in, stab.data(), sizeof(double) * stab.size()))
    return 2;
  const int r = precision == 0 ? run<double>(in, out, mp, nsteps, dels, glob, vtab, stab)
                               : run<float>(in, out, mp, nsteps, dels, glob, vtab, stab);
  fclose(in);
  fclose(out);
  return r;
}
