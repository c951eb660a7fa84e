// engine_fft64.hip -- mesh transforms of FP64 fields.
#include "engine_fft.hpp"

namespace trvg {

#define TRVG_COMMA ,
#define TRVG_FFT3D_INST(L)                                                        \
  template void fft3d<double, L>(Context&, c2<double>*, const L&, int, double, const Prune*);
TRVG_FFT3D_INST(LoadSame<double>)
TRVG_FFT3D_INST(LoadScaleShift<double>)
TRVG_FFT3D_INST(LoadLinear2<double>)
TRVG_FFT3D_INST(LoadTwopt<double TRVG_COMMA double>)
TRVG_FFT3D_INST(LoadTwopt<double TRVG_COMMA double TRVG_COMMA true>)
TRVG_FFT3D_INST(LoadDeconv<double TRVG_COMMA double>)
// Loaders of the differentiable path (engine_diff.hip).
TRVG_FFT3D_INST(LoadReal<double>)
TRVG_FFT3D_INST(LoadShell<double TRVG_COMMA double>)
#undef TRVG_FFT3D_INST

template void shell_slab_work<double>(const Geom&, const trvg_binning&, int, int, bool,
                                   std::vector<ShellBand>&, std::vector<double>&,
                                   std::vector<int2>&, std::vector<int2>&,
                                   std::vector<int2>&);
template void shell_slab_ifft<double, double>(Context&, c2<double>*, const double2*,
                                           const trvg_binning&, const std::vector<int>&,
                                           const std::vector<int>&, int, int, bool);
template void slab_fft<double>(Context&, c2<double>*, int);
template void full_work<double>(const Geom&, int, std::vector<int2>&, std::vector<int2>&,
                             std::vector<int2>&);
template void sjl_slab_ifft<double>(Context&, c2<double>*, const double2*, const Spline&,
                                 const std::vector<double>&, const std::vector<int>&, int, int,
                                 bool);

// Batched plans (engine_batch.hip).
#define TRVG_FFT3D_BATCH_INST(L)                                                  \
  template void fft3d_batch<double, L>(Context&, c2<double>*, const L&, int, bool,      \
                                    const double*, const int2*, int, const int2*, \
                                    int, const int2*, int);
TRVG_FFT3D_BATCH_INST(LoadScaleShiftMocks)
TRVG_FFT3D_BATCH_INST(LoadTwoptMocks)
TRVG_FFT3D_BATCH_INST(LoadShellMocks<double>)
TRVG_FFT3D_BATCH_INST(LoadShellPairMocks<double>)
TRVG_FFT3D_BATCH_INST(LoadDeconvMocks<double>)

}  // namespace trvg
