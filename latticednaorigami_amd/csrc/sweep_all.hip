// sweep_all.hip - sweep kernels for movesets with recoil-growth or jump moves.
#include <hip/hip_runtime.h>

#define LDO_SWEEP_WAVE_KERNELS
#include "sweep_wave.h"

WaveKernels wave_kernels_all() {
    return WaveKernels {ldo_sweep_lds_kernel<true>, ldo_batch_sweep_lds_kernel<true>};
}
