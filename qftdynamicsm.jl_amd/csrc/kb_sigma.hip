// kb_sigma.hip -- self-energy stage (kb_sigma_impl.h): what is common to the
// modes, and the choice of the form.
#include <mutex>

#include "kb_sigma_impl.h"

namespace qftkb {

namespace {

constexpr int SIGMA_DEVICES = 64;  // (further ones are prepared at every call)
constexpr int FORMS[] = {FORM_FLAT, FORM_WHOLE, FORM_PASSES, PLAN_SMALL, PLAN_ANY, PLAN_WIDE};
constexpr int NFORMS = 6, NMODES = SG_PLAIN + 1;

struct FormCode {
  hipError_t (*launch)(const SigmaArgs&, int, int, hipStream_t);
  hipError_t (*prepare)();
};

}  // namespace

#define KB_FORM(MODE, FORM)                                                            \
  template <>                                                                          \
  hipError_t sigma_form<MODE, FORM>(const SigmaArgs&, int rows, int want, hipStream_t st); \
  template <>                                                                          \
  hipError_t sigma_form_prepare<MODE, FORM>();
#define KB_MODE(MODE)                                                                \
  KB_FORM(MODE, FORM_FLAT) KB_FORM(MODE, FORM_WHOLE) KB_FORM(MODE, FORM_PASSES)      \
  KB_FORM(MODE, PLAN_SMALL) KB_FORM(MODE, PLAN_ANY) KB_FORM(MODE, PLAN_WIDE)
KB_MODE(SG_SUNSET)
KB_MODE(SG_SUNSET_ADJ)
KB_MODE(SG_BUBBLE)
KB_MODE(SG_CHAIN)
KB_MODE(SG_PLAIN)
#undef KB_MODE
#undef KB_FORM

namespace {

// (in the order of SigmaMode and of FORMS)
#define KB_FORM(MODE, FORM) {sigma_form<MODE, FORM>, sigma_form_prepare<MODE, FORM>}
#define KB_MODE(MODE)                                                                 \
  {KB_FORM(MODE, FORM_FLAT),  KB_FORM(MODE, FORM_WHOLE), KB_FORM(MODE, FORM_PASSES),  \
   KB_FORM(MODE, PLAN_SMALL), KB_FORM(MODE, PLAN_ANY),   KB_FORM(MODE, PLAN_WIDE)}
const FormCode kForms[NMODES][NFORMS] = {KB_MODE(SG_SUNSET), KB_MODE(SG_SUNSET_ADJ), KB_MODE(SG_BUBBLE),
                                         KB_MODE(SG_CHAIN), KB_MODE(SG_PLAIN)};
#undef KB_MODE
#undef KB_FORM

int form_index(int form) {
  int i = 0;
  while (FORMS[i] != form) ++i;
  return i;
}

}  // namespace

void plan_fft(FFTPlan& pl, int n) { pl = make_plan(n); }

// A first call on a device also loads the form's code there (1 to 2 ms; all of it
// took 13 ms of a process's first kb_create), so only what a lattice runs is
// prepared.
hipError_t sigma_prepare(SigmaMode mode, int Nx, int sdim, int device) {
  static std::mutex mu;
  static bool ready[SIGMA_DEVICES][NMODES][NFORMS] = {};
  bool used[NFORMS] = {};
  if (Nx > 0) {
    const FFTPlan pl = make_plan(Nx);
    for (int rows : {1, SPREAD_ROWS}) used[form_index(stage_form(pl, sdim, rows, true))] = true;
  }
  std::lock_guard<std::mutex> lk(mu);
  const bool known = device >= 0 && device < SIGMA_DEVICES;
  for (int f = 0; f < NFORMS; ++f) {
    if ((Nx > 0 && !used[f]) || (known && ready[device][mode][f])) continue;
    const hipError_t e = kForms[mode][f].prepare();
    if (e != hipSuccess) return e;
    if (known) ready[device][mode][f] = true;
  }
  return hipSuccess;
}

// (3D rows that a workgroup holds whole do without; the workspace is part of
// what a 3D context holds all the same)
size_t sigma_workspace_values(int Nx, int sdim, size_t rows) {
  if (sdim == 1 || (sdim == 2 && planes_fit(Nx))) return 0;
  return rows * (sdim == 3 ? (size_t)Nx * Nx : (size_t)Nx) * (Nx / 2 + 1);
}

// whole planes of up to 64 x 64 points, 1D lattices up to 2048: the sizes
// whose stage serves orbit storage through its site maps
bool sigma_planes_supported(int Nx, int sdim) { return Nx >= 1 && Nx <= (sdim == 1 ? 2048 : 64); }

// threads per workgroup the autotuner asks for (run-time plans of planes and
// batches); entry 0 is the default.  A step's stage with 24 rows, us, for 256,
// 128 and 512: 27^3 34 34 34, 35^3 39 48 39, 45^3 54 70 53, 50^3 65 73 76, 46^3
// 116 122 137, 57^3 146 133 151, 63^3 128 131 113, 61^3 275 297 201.
const int kFFTThreads[NFFT_VARIANTS] = {256, 128, 512, 1024};

hipError_t launch_sigma_stage(const SigmaArgs& a, SigmaMode mode, int rows, hipStream_t st, int variant, bool alone) {
  const int form = stage_form(a.plan, a.ny == 1 ? 1 : a.nz == 1 ? 2 : 3, rows, alone);
  return kForms[mode][form_index(form)].launch(a, rows, kFFTThreads[variant], st);
}

}  // namespace qftkb
