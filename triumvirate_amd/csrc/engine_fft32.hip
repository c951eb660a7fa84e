// engine_fft32.hip -- mesh transforms of FP32 fields.
#include "engine_fft.hpp"

namespace trvg {

#define TRVG_COMMA ,
#define TRVG_FFT3D_INST(L)                                                        \
  template void fft3d<float, L>(Context&, c2<float>*, const L&, int, double, const Prune*);
TRVG_FFT3D_INST(LoadSame<float>)
TRVG_FFT3D_INST(LoadTwopt<float TRVG_COMMA double>)
TRVG_FFT3D_INST(LoadDeconv<float TRVG_COMMA double>)
// Loaders of the differentiable path (engine_diff.hip).
TRVG_FFT3D_INST(LoadReal<float>)
TRVG_FFT3D_INST(LoadDeconv<float TRVG_COMMA float>)
TRVG_FFT3D_INST(LoadShell<float TRVG_COMMA float>)
#undef TRVG_FFT3D_INST

template void shell_slab_work<float>(const Geom&, const trvg_binning&, int, int, bool,
                                   std::vector<ShellBand>&, std::vector<double>&,
                                   std::vector<int2>&, std::vector<int2>&,
                                   std::vector<int2>&);
template void shell_slab_ifft<float, double>(Context&, c2<float>*, const double2*,
                                           const trvg_binning&, const std::vector<int>&,
                                           const std::vector<int>&, int, int, bool);
template void shell_slab_ifft<float, float>(Context&, float2*, const float2*,
                                            const trvg_binning&, const std::vector<int>&,
                                            const std::vector<int>&, int, int, bool);
template void slab_fft<float>(Context&, c2<float>*, int);
template void full_work<float>(const Geom&, int, std::vector<int2>&, std::vector<int2>&,
                             std::vector<int2>&);
template void sjl_slab_ifft<float>(Context&, c2<float>*, const double2*, const Spline&,
                                 const std::vector<double>&, const std::vector<int>&, int, int,
                                 bool);

// Batched plans (engine_batch.hip).
#define TRVG_FFT3D_BATCH_INST(L)                                                  \
  template void fft3d_batch<float, L>(Context&, c2<float>*, const L&, int, bool,      \
                                    const double*, const int2*, int, const int2*, \
                                    int, const int2*, int);
TRVG_FFT3D_BATCH_INST(LoadShellMocks<float>)
TRVG_FFT3D_BATCH_INST(LoadShellPairMocks<float>)
TRVG_FFT3D_BATCH_INST(LoadDeconvMocks<float>)

}  // namespace trvg
