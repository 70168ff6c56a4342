// Device helpers of the folded contractions (op_kernels.hip, contract_block.h,
// contract_direct.hip) and of the Hankel filter (green_assembly.hip): waits on copies in
// flight, the 16x16x4 MFMAs and their lane layout, LDS reads by byte offset.
#pragma once

#include "xtr_common.h"

namespace xtr {

template <int N>
__device__ __forceinline__ void wait_vm()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS writes of this wave (partial sums) must be complete before other waves pass the barrier and
// read them: s_barrier alone does not wait for them.
#define XTR_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

typedef double mfma_d4 __attribute__((ext_vector_type(4)));
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
template <typename T> struct MfmaAcc;
template <> struct MfmaAcc<double> { typedef mfma_d4 type; };
template <> struct MfmaAcc<float> { typedef mfma_f4 type; };
__device__ __forceinline__ mfma_d4 mfma16(double a, double b, mfma_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mfma_f4 mfma16(float a, float b, mfma_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// Row of D held in register r of lane l (16x16x4 results; column = l % 16): the FP64 instruction
// spreads consecutive rows over the lane quarters, the FP32 one over the registers.
template <typename T>
__device__ __forceinline__ int mfma_row(int lane, int r)
{
    return sizeof(T) == 8 ? 4 * r + (lane >> 4) : 4 * (lane >> 4) + r;
}

// D += (NEG ? -a : a) b. The FP64 instruction negates its A operand itself (the neg modifier);
// the FP32 one has no such modifier, the sign goes on the value.
template <bool NEG>
__device__ __forceinline__ mfma_d4 mfma16s(double a, double b, mfma_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, NEG ? 1 : 0);
}
template <bool NEG>
__device__ __forceinline__ mfma_f4 mfma16s(float a, float b, mfma_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -a : a, b, c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ cplx<T> lds_cplx(const cplx<T> *blk, unsigned off)
{
    return *reinterpret_cast<const cplx<T> *>(reinterpret_cast<const char *>(blk) + off);
}
template <typename T>
__device__ __forceinline__ T lds_part(const cplx<T> *blk, unsigned off)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(blk) + off);
}

}  // namespace xtr
