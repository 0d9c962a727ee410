// What the two batched GEMM translation units share: the launch record, the
// weight unpacking and the epilogue expressions.
#pragma once
#include <cmath>

#include "vgx_internal.h"
#include "vgx_qrow.h"

#pragma clang fp contract(off)

enum BatchEpi { BEPI_STORE = 0, BEPI_GATE = 1, BEPI_SPLIT = 2 };

struct GemmLaunch {
    MatDev M, M3;           // W (and W3 for the gate)
    int ntok, cols;
    const int16_t* x;       // ntok rows of cols q16 values, row stride ldx
    int ldx;
    const int16_t* res;     // residual rows (stride ldy) or nullptr
    int16_t* y;             // ntok rows of M.rows q16 values, row stride ldy
    int ldy;
    int hs;                 // gate: hidden store exponent
    int split;              // split: first column of the second half
    const int16_t* rw;      // RMS prologue: the q16 norm weight (cols values)
    float eps;              // RMS prologue: epsilon
    long long* part;        // split K: [split][set][ntok][rows] exact partial sums
    int nz;                 // split K: the launch's splits (its grid's z; from here, not from
                            // gridDim.z, an implicit argument whose load would delay the first weights)
};

// The tile kernel of vgx_gemm.hip; VGX_ESTATE past its limits on rows and grid.
int vgx_gemm_tile_launch(const GemmLaunch& L, int epi, int num_cu, hipStream_t s);

namespace {

typedef signed char i8x16 __attribute__((ext_vector_type(16)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int kTile = 32;  // tokens and weight rows of a matrix-core tile

union Op {
    i8x16 v;
    uint32_t d[4];
};

__device__ __forceinline__ i32x16 mfma(const Op& a, const Op& b, const i32x16& c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a.v, b.v, c, 0, 0, 0);
}

// Four 2-bit t3 codes (one byte, code j at bits 2j..2j+1) as four int8
// levels: bit 0 = |level|, bit 1 = sign (engine/tools/mmcf_hf.py:168-199);
// code 2 (a sign without magnitude) is level 0.  Each code is spread to its
// own byte, then level = |l| ^ ((sign & |l|) * 0xFE): 0x01 or 0xFF.
__device__ __forceinline__ uint32_t t3_levels(uint32_t b) {
    const uint32_t x = (b | (b << 6) | (b << 12) | (b << 18)) & 0x03030303u;
    const uint32_t m = x & 0x01010101u;
    const uint32_t sg = (x >> 1) & m;
    return m ^ (sg * 0xFEu);
}

__device__ __forceinline__ float gate_value(float v1, float v3, int hs) {
    const float g = (float)q16_round(v1), uu = (float)q16_round(v3);
    const float a = g / 256.0f;
    const float e = (float)exp(-(double)a);
    const float dn = 1.0f + e;
    const float r = a / dn;
    float o = r * (uu / 256.0f);
    o = o * ldexpf(1.0f, -hs);
    return o * 256.0f;
}

}  // namespace
