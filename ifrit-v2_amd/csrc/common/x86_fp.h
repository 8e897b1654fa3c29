// x86 SSE/AVX floating-point semantics needed to reproduce the tile
// rasterizer's CPU arithmetic bit for bit on gfx950.
//
// The CPU path (projects/softgraphics/src/engine/tileraster/TileRasterWorker.cpp)
// is written with SSE/AVX2 intrinsics whose results differ from plain IEEE
// C math in four places, each emulated here:
//   * RCPPS / RCPSS, the 12-bit reciprocal approximation
//     (include/ifrit/core/math/fastutil/FastUtilSimd.h:27-33, 87-97), whose
//     outputs differ between CPU vendors: a table for Intel and one for AMD;
//   * MINPS / MAXPS, which return the second operand when the comparison is
//     false (NaN or equal operands), unlike fminf/fmaxf;
//   * CVTTSS2SI, which returns INT_MIN for NaN and out-of-range inputs
//     where the GPU conversion saturates (TileRasterWorker.cpp:319-322);
//   * DPPS, which sums ((p0 + p1) + (p2 + p3)) with masked products as +0
//     (include/ifrit/core/math/simd/SimdVectors.h:497-510).
// Everything else is IEEE single precision with round-to-nearest-even; the
// kernels are compiled with -ffp-contract=off and call fmaf where the CPU
// code calls an FMA intrinsic.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define IFX_HD __host__ __device__ __forceinline__
#else
#include <math.h>
#include <string.h>
#define IFX_HD static inline
#endif

namespace ifx {

// Whose RCPSS to reproduce.  The instruction is implementation-defined: on
// the Intel CPU its table was captured on the result depends on the top 11
// mantissa bits, on the AMD EPYC its other table was captured on, on the top
// 12; both scale exactly with the exponent and share the special cases.
enum RcpModel : int { kRcpIntel = 0, kRcpAmd = 1 };

#if defined(__HIPCC__)
__device__ __constant__ static const uint32_t kRcpTable[2048] = {
#include "x86_rcp_table.inc"
};
__device__ __constant__ static const uint32_t kRcpTableAmd[4096] = {
#include "x86_rcp_table_amd.inc"
};
#endif
// Host copies of the same data for host-side setup code.
static const uint32_t kRcpTableHost[2048] = {
#include "x86_rcp_table.inc"
};
static const uint32_t kRcpTableAmdHost[4096] = {
#include "x86_rcp_table_amd.inc"
};

IFX_HD uint32_t f2u(float f) { return __builtin_bit_cast(uint32_t, f); }
IFX_HD float u2f(uint32_t u) { return __builtin_bit_cast(float, u); }

// RCPSS/RCPPS of the given model: table lookup on the top 11 (Intel) or 12
// (AMD) mantissa bits, exact exponent scaling, sub-normal results flushed to
// signed zero, zero and sub-normal inputs give signed infinity, infinities
// give signed zero, NaNs come back quieted.
// Without branches: the table's entry for the mantissa with 127 - e added to its
// exponent, replaced where that leaves the normal range.
// In three steps, so that a caller can have several lookups in flight.
struct RcpTable {
    const uint32_t* entries;
    uint32_t shift, mask;
};
IFX_HD RcpTable rcp_table(int model) {
    const bool amd = model == kRcpAmd;
#if defined(__HIP_DEVICE_COMPILE__)
    return RcpTable{amd ? kRcpTableAmd : kRcpTable, amd ? 11u : 12u, amd ? 0xfffu : 0x7ffu};
#else
    return RcpTable{amd ? kRcpTableAmdHost : kRcpTableHost, amd ? 11u : 12u, amd ? 0xfffu : 0x7ffu};
#endif
}
IFX_HD uint32_t rcp_entry(float x, const RcpTable& tab) { return tab.entries[(f2u(x) >> tab.shift) & tab.mask]; }
IFX_HD float rcp_ps(float x, uint32_t entry) {
    const uint32_t b = f2u(x);
    const uint32_t sign = b & 0x80000000u;
    const int32_t e = (int32_t)((b >> 23) & 0xffu);
    const int32_t t = (int32_t)entry + ((127 - e) * 0x800000);  // exponents 126 or 127 in the table
    uint32_t r = t < 0x800000 ? 0u : (uint32_t)t;                  // sub-normal results flush to zero
    r = e == 0 ? 0x7f800000u : r;
    r = e == 255 ? ((b & 0x7fffffu) ? (b & 0x7fffffffu) | 0x400000u : 0u) : r;
    return u2f(sign | r);
}
IFX_HD float rcp_ps(float x, int model) { return rcp_ps(x, rcp_entry(x, rcp_table(model))); }

// ApproxReciprocalNR256: r = rcp(x); (r + r) - x * (r * r).
IFX_HD float rcp_nr_ps(float x, uint32_t entry) {
    float r = rcp_ps(x, entry);
    float rr = r * r;
    float muls = x * rr;
    float twice = r + r;
    return twice - muls;
}

// ApproxReciprocal (scalar): r = rcp(x); r * (2 - r * x).
IFX_HD float rcp_nr_ss(float x, int model) {
    float r = rcp_ps(x, model);
    float rx = r * x;
    float t = 2.0f - rx;
    return r * t;
}

IFX_HD float min_ps(float a, float b) { return a < b ? a : b; }
IFX_HD float max_ps(float a, float b) { return a > b ? a : b; }

// CVTTSS2SI: truncation toward zero; 0x80000000 when NaN or out of range.
IFX_HD int cvtt_i32(float x) {
    if (!(x > -2147483904.0f && x < 2147483648.0f)) return (int)0x80000000u;
    return (int)x;
}

IFX_HD float neg(float x) { return u2f(f2u(x) ^ 0x80000000u); }

}  // namespace ifx
