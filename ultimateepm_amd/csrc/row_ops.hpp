// row_ops.hpp — multiply-adds whose second factor sits in another lane of the
// same 16-lane DPP row (gfx950): v_fmac_*_dpp row_newbcast:r multiplies by the
// value that lane r of each row holds, so sixteen factors shared by a row cost
// one register per lane and no move.  Measured issue intervals of one SIMD (four
// waves, cycles per wave instruction): v_fmac_f32 2.8, v_fmac_f32_dpp 4.7,
// v_fmac_f64 and v_fmac_f64_dpp 4.8: the DPP operand is free in FP64.
// Plain VALU instructions; each block opens with the two wait states a DPP
// operand needs after a VALU write.
// The accumulators are early clobbers: several instructions write them while later
// ones still read the factors, so none may share a register with a factor of the
// same value (it may where the compiler sees the two equal, as in a first pass over zeros).
#pragma once
#include <hip/hip_runtime.h>

namespace uepm {
namespace rowop {

#define UEPM_MV(T, a, m, r) \
    "v_fmac_" T "_dpp %" a ", %4, %" m " row_newbcast:" r " row_mask:0xf bank_mask:0xf\n\t"
#define UEPM_MV16(T)                                                                                             \
    "s_nop 1\n\t" UEPM_MV(T, "0", "5", "0") UEPM_MV(T, "1", "6", "1") UEPM_MV(T, "2", "7", "2")                \
        UEPM_MV(T, "3", "8", "3") UEPM_MV(T, "0", "9", "4") UEPM_MV(T, "1", "10", "5") UEPM_MV(T, "2", "11", "6") \
            UEPM_MV(T, "3", "12", "7") UEPM_MV(T, "0", "13", "8") UEPM_MV(T, "1", "14", "9")                     \
                UEPM_MV(T, "2", "15", "10") UEPM_MV(T, "3", "16", "11") UEPM_MV(T, "0", "17", "12")              \
                    UEPM_MV(T, "1", "18", "13") UEPM_MV(T, "2", "19", "14") UEPM_MV(T, "3", "20", "15")
#define UEPM_MV_OPS                                                                                              \
    : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3])                                                 \
    : "v"(v), "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(A[4]), "v"(A[5]), "v"(A[6]), "v"(A[7]), "v"(A[8]), \
      "v"(A[9]), "v"(A[10]), "v"(A[11]), "v"(A[12]), "v"(A[13]), "v"(A[14]), "v"(A[15])

// acc[r % 4] += A[r] * (v of lane r of the row), r = 0..15
__device__ __forceinline__ void dot16(float (&acc)[4], float v, const float (&A)[16]) {
    asm(UEPM_MV16("f32") UEPM_MV_OPS);
}
__device__ __forceinline__ void dot16(double (&acc)[4], double v, const double (&A)[16]) {
    asm(UEPM_MV16("f64") UEPM_MV_OPS);
}

#define UEPM_AX(T, a, r) "v_fmac_" T "_dpp %" a ", %8, %9 row_newbcast:" r " row_mask:0xf bank_mask:0xf\n\t"
#define UEPM_AX8(T, r0, r1, r2, r3, r4, r5, r6, r7)                                                              \
    "s_nop 1\n\t" UEPM_AX(T, "0", r0) UEPM_AX(T, "1", r1) UEPM_AX(T, "2", r2) UEPM_AX(T, "3", r3)              \
        UEPM_AX(T, "4", r4) UEPM_AX(T, "5", r5) UEPM_AX(T, "6", r6) UEPM_AX(T, "7", r7)
#define UEPM_AX_OPS(o)                                                                                           \
    : "+&v"(A[o]), "+&v"(A[o + 1]), "+&v"(A[o + 2]), "+&v"(A[o + 3]), "+&v"(A[o + 4]), "+&v"(A[o + 5]),         \
      "+&v"(A[o + 6]), "+&v"(A[o + 7])                                                                           \
    : "v"(x), "v"(c)

// A[r] += c * (x of lane r of the row), r = 0..15
__device__ __forceinline__ void axpy16(float (&A)[16], float x, float c) {
    asm(UEPM_AX8("f32", "0", "1", "2", "3", "4", "5", "6", "7") UEPM_AX_OPS(0));
    asm(UEPM_AX8("f32", "8", "9", "10", "11", "12", "13", "14", "15") UEPM_AX_OPS(8));
}
__device__ __forceinline__ void axpy16(double (&A)[16], double x, double c) {
    asm(UEPM_AX8("f64", "0", "1", "2", "3", "4", "5", "6", "7") UEPM_AX_OPS(0));
    asm(UEPM_AX8("f64", "8", "9", "10", "11", "12", "13", "14", "15") UEPM_AX_OPS(8));
}
#undef UEPM_MV
#undef UEPM_MV16
#undef UEPM_MV_OPS
#undef UEPM_AX
#undef UEPM_AX8
#undef UEPM_AX_OPS

}  // namespace rowop
}  // namespace uepm
