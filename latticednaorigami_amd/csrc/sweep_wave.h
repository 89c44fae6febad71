// sweep_wave.h - the sweep kernels on the wavefront engine.
//
// Two kernels each, for movesets with and without recoil-growth and jump
// moves (ALL), in a source file of its own: their code is four times that of
// the standard moveset's and would sit between its parts.
#ifndef LDO_SWEEP_WAVE_H
#define LDO_SWEEP_WAVE_H

#include "replica_ops.h"

typedef void (*SweepFn)(Params, int64_t, const int32_t*, const int32_t*);
typedef void (*BatchSweepFn)(const Params*, const int32_t*, int32_t, int64_t);
struct WaveKernels {
    SweepFn sweep;
    BatchSweepFn batch;
};
WaveKernels wave_kernels_std(); // sweep_std.hip
WaveKernels wave_kernels_all(); // sweep_all.hip
inline WaveKernels wave_kernels(const Params& P) {
    return wave_all_kinds(P) ? wave_kernels_all() : wave_kernels_std();
}

// The replica a workgroup of the one-replica-per-workgroup sweeps runs.
// Workgroups are dealt to the 8 XCDs round-robin, so workgroup b runs on XCD
// b % 8; when the ladder divides into 8 equal runs of slots, XCD x takes the
// replicas of slots [x R/8, (x+1) R/8), so that each XCD's L2 holds the
// energy tables of few temperatures (slots are temperature-major).  q_to_rep
// (slot -> replica) is the exchange's permutation, or null for the identity.
__device__ __forceinline__ int replica_of_block(const Params& P, const int32_t* q_to_rep) {
    int b = blockIdx.x, R = P.n_replicas;
    int q = (R % 8 == 0) ? (b % 8) * (R / 8) + b / 8 : b;
    return q_to_rep != nullptr ? q_to_rep[q] : q;
}

#ifdef LDO_SWEEP_WAVE_KERNELS
// One wavefront per replica with the wavefront engine (engine_wave.h): the
// staged part of the block is copied to LDS, the chain runs there and the
// block is written back.  The host picks this kernel where wave_lds_bytes(P)
// of dynamic LDS fit.
template <bool ALL>
__device__ __forceinline__ void sweep_staged(const Params& P, int r, char* blk, lds_t lds,
                                             int64_t steps, const int32_t* rep_slot) {
    int n16 = (int)(P.L.stage / 16);
    Quad* g = (Quad*)blk;
    LDO_LDS Quad* l = (LDO_LDS Quad*)lds;
    int lane = threadIdx.x & 63;
    for (int i = lane; i < n16; i += 64) {
        l[i] = g[i];
    }
    sweep_wave<ALL>(P, r, blk, lds, steps, rep_slot);
    for (int i = lane; i < n16; i += 64) {
        g[i] = l[i];
    }
}

template <bool ALL>
__global__ void __launch_bounds__(64)
    ldo_sweep_lds_kernel(Params P, int64_t steps, const int32_t* rep_slot,
                         const int32_t* q_to_rep) {
    extern __shared__ Quad lds_block[];
    if ((int)blockIdx.x >= P.n_replicas) {
        return;
    }
    int r = uni(replica_of_block(P, q_to_rep));
    sweep_staged<ALL>(P, r, P.blocks + (size_t)r * P.L.bytes, (lds_t)lds_block, steps, rep_slot);
}

// One wavefront per chain of `order` (n of them) with the wavefront engine;
// dynamic LDS = the largest wave_lds_bytes of these chains.
template <bool ALL>
__global__ void __launch_bounds__(64)
    ldo_batch_sweep_lds_kernel(const Params* plist, const int32_t* order, int32_t n,
                               int64_t steps) {
    extern __shared__ Quad lds_block[];
    if ((int)blockIdx.x >= n) {
        return;
    }
    int k = uni(order[blockIdx.x]);
    // nothing writes the parameters during a launch: scalar loads
    const Params& P = *(const Params*)(__attribute__((address_space(4))) const Params*)(plist + k);
    sweep_staged<ALL>(P, 0, P.blocks, (lds_t)lds_block, steps, nullptr);
}
#endif // LDO_SWEEP_WAVE_KERNELS

#endif
