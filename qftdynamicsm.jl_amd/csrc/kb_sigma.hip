// kb_sigma.hip -- self-energy stage (kb_sigma_impl.h): the sunset's passes and
// what is common to the modes.
#include "kb_sigma_impl.h"

namespace qftkb {

KB_SIGMA_MODE(SG_SUNSET)

void plan_fft(FFTPlan& pl, int n) { pl = make_plan(n); }

hipError_t sigma_prepare() {
  hipError_t e = sigma_prepare_mode<SG_SUNSET>();
  if (e == hipSuccess) e = sigma_prepare_mode<SG_SUNSET_ADJ>();
  if (e == hipSuccess) e = sigma_prepare_mode<SG_BUBBLE>();
  if (e == hipSuccess) e = sigma_prepare_mode<SG_CHAIN>();
  if (e == hipSuccess) e = sigma_prepare_mode<SG_PLAIN>();
  return e;
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

// threads per workgroup the autotuner asks for; entry 0 is the default
const int kFFTThreads[NFFT_VARIANTS] = {256, 128, 512, 1024};

hipError_t launch_sigma_stage(const SigmaArgs& a, SigmaMode mode, int rows, hipStream_t st, int variant) {
  const int want = kFFTThreads[variant];
  switch (mode) {
    case SG_SUNSET: return sigma_stage<SG_SUNSET>(a, rows, want, st);
    case SG_SUNSET_ADJ: return sigma_stage<SG_SUNSET_ADJ>(a, rows, want, st);
    case SG_BUBBLE: return sigma_stage<SG_BUBBLE>(a, rows, want, st);
    case SG_CHAIN: return sigma_stage<SG_CHAIN>(a, rows, want, st);
    default: return sigma_stage<SG_PLAIN>(a, rows, want, st);
  }
}

}  // namespace qftkb
