// sweep_std.hip - sweep kernels for the standard moveset: orientation rotation, staple exchange,
// CB staple and CTCB scaffold regrowth.
#include <hip/hip_runtime.h>

#define LDO_SWEEP_WAVE_KERNELS
#include "sweep_wave.h"

WaveKernels wave_kernels_std() {
    return WaveKernels {ldo_sweep_lds_kernel<false>, ldo_batch_sweep_lds_kernel<false>};
}
