// Device-side reductions shared by the kernel files.  Their summation order
// is part of the results: the fused loop kernels (cmbl_loops.hip) replicate
// the plain dot product (k_dot_part + k_dot_final) exactly through them.
#pragma once

#include <hip/hip_runtime.h>

namespace cmbl {

// A wave-uniform value that the kernel itself stores to later.  A plain load of
// it may become a scalar load, which is not ordered with the wave's vector
// stores: a store issued after it can reach memory first.  Atomic loads go
// through vector memory, in order with them.
template <class T>
__device__ __forceinline__ T load_before_store(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Lanes 0..31 get a summed over lanes (j, j + 32), lanes 32..63 get b summed
// likewise (v_permlane32_swap exchanges lanes 32..63 of its first operand
// with lanes 0..31 of its second).
__device__ __forceinline__ double swap32_add(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b),
                                                     false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Rows of 16 lanes: rows 0 and 2 get a summed over row pairs (0,1) and (2,3),
// rows 1 and 3 get b summed likewise (v_permlane16_swap exchanges the odd rows
// of its first operand with the even rows of its second).
__device__ __forceinline__ double swap16_add(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b),
                                                     false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// s plus s rotated by N lanes within each row of 16 (DPP row_ror:N); for
// N = 8 that is s plus s of lane j ^ 8.
template <int N>
__device__ __forceinline__ double ror_add(double s)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(s), 0x120 + N, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(s), 0x120 + N, 0xF, 0xF, false);
    return s + __hiloint2double(hi, lo);
}

// Sum over the 64 lanes of a wavefront (butterfly; every lane gets the sum).
__device__ __forceinline__ double wave_sum(double v)
{
    // lane j adds lane j ^ o for o = 32, 16, .., 1; from o = 8 on the values have
    // period 2 o in a row, where a rotation by o is the exchange (moves in the
    // VALU: by LDS permutes a sum took 12 of them, 0.3 us alone)
    v = swap32_add(v, v);
    v = swap16_add(v, v);
    v = ror_add<8>(v);
    v = ror_add<4>(v);
    v = ror_add<2>(v);
    return ror_add<1>(v);
}

// Block-wide sum for blockDim.x == NT (multiple of 64): wave sums, then
// thread 0 adds them in wave order starting from 0.  Result valid in thread 0.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double* sh)
{
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0) {
        for (int i = 0; i < NT / 64; ++i) t += sh[i];
    }
    __syncthreads();
    return t;
}

}  // namespace cmbl
