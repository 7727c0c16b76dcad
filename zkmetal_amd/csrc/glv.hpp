// Scalar side of the MSM on the device: reduction mod r, the GLV split
// k == (+-k1) + lambda*(+-k2) (mod r) of Sources/zkMetal/MSM/GLV.swift:37-92 /
// Sources/Shaders/msm/glv_kernels.metal:172-256 (same lattice constants and
// truncated Babai rounding), and the signed c-bit recoding of
// Sources/Shaders/msm/msm_kernels.metal:399-439.
//
// Bounds (checked numerically from the constants): c1*a2 < r, so one
// conditional "+r" after each subtraction keeps k1 in [0, r); the folded
// |k1| and |k2| are below 2^126.97, so ceil(128/c) signed windows never leave
// a final carry (the kernel still reports one as an error).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zk {

// r = 0x30644e72e131a029b85045b68181585d2833e84879b9709143e1f593f0000001
__device__ __forceinline__ uint32_t r_limb(int i) {
    switch (i) {
        case 0: return 0xf0000001u;
        case 1: return 0x43e1f593u;
        case 2: return 0x79b97091u;
        case 3: return 0x2833e848u;
        case 4: return 0x8181585du;
        case 5: return 0xb85045b6u;
        case 6: return 0xe131a029u;
        default: return 0x30644e72u;
    }
}

// Fr element in Montgomery form (x * 2^256 mod r, the reference's Fr limbs)
// -> standard form x, for any 256-bit input: Montgomery reduction REDC(k),
// the same value as the reference's fr_mul(k, 1)
// (Sources/NeonFieldOps/bn254_msm.c:1537-1552).  The REDC result is below
// r + 1, so one conditional subtraction makes it canonical.
#define ZK_RINV32 0xefffffffu  // -r^-1 mod 2^32
__device__ __forceinline__ void fr_from_mont(uint32_t k[8]) {
    uint32_t t[17];
#pragma unroll
    for (int i = 0; i < 8; i++) t[i] = k[i];
#pragma unroll
    for (int i = 8; i < 17; i++) t[i] = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t m = t[i] * ZK_RINV32;  // t + m r == 0 mod 2^(32(i+1))
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint64_t s = (uint64_t)m * r_limb(j) + t[i + j] + c;
            t[i + j] = (uint32_t)s;
            c = s >> 32;
        }
#pragma unroll
        for (int j = i + 8; j < 17; j++) {
            const uint64_t s = (uint64_t)t[j] + c;
            t[j] = (uint32_t)s;
            c = s >> 32;
        }
    }
    uint32_t d[8];
    unsigned br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) d[i] = __builtin_subc(t[8 + i], r_limb(i), br, &br);
    br = (t[16] == 0) ? br : 0u;  // t[16] is 0: the result is < r + 1 < 2^256
#pragma unroll
    for (int i = 0; i < 8; i++) k[i] = br ? t[8 + i] : d[i];
}

// out[0..na+nb) = a[0..na) * b[0..nb)
template <int NA, int NB>
__device__ __forceinline__ void mul_wide(const uint32_t* a, const uint32_t* b, uint32_t* out) {
#pragma unroll
    for (int i = 0; i < NA + NB; i++) out[i] = 0;
#pragma unroll
    for (int i = 0; i < NA; i++) {
        uint32_t carry = 0;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            uint64_t t = (uint64_t)a[i] * b[j] + out[i + j] + carry;
            out[i + j] = (uint32_t)t;
            carry = (uint32_t)(t >> 32);
        }
        out[i + NB] = carry;
    }
}

// a -= b over N limbs; returns the borrow
template <int N>
__device__ __forceinline__ unsigned sub_n(uint32_t* a, const uint32_t* b) {
    unsigned br = 0;
#pragma unroll
    for (int i = 0; i < N; i++) a[i] = __builtin_subc(a[i], b[i], br, &br);
    return br;
}

__device__ __forceinline__ bool geq_r(const uint32_t* a) {
    unsigned br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) (void)__builtin_subc(a[i], r_limb(i), br, &br);
    return br == 0;
}

struct GlvSplit {
    uint32_t k1[4], k2[4];
    bool neg1, neg2;
};

// Words FROM.. of a * b (NA and NB words, b uniform), column by column; the
// products of lower columns are left out, so out[FROM] is low by less than
// min(NA, NB) carries into the column above, which is why the caller starts
// one column early and looks.  LAST: words past it are not wanted.
template <int NA, int NB, int FROM, int LAST>
__device__ __forceinline__ void mul_columns(const uint32_t* a, const uint32_t* b, uint32_t* out) {
    uint64_t lo = 0;
#pragma unroll
    for (int q = FROM; q <= LAST; q++) {
        uint32_t hi = 0;
        const int end = q < NA ? q + 1 : NA;  // i < end, q - i < NB
        int i = q < NB ? 0 : q - NB + 1;
        if (q < LAST) {
#pragma unroll
            for (; i + 3 <= end; i += 3)
                mac_uniform(lo, hi, a[i], b[q - i], a[i + 1], b[q - i - 1], a[i + 2], b[q - i - 2]);
            if (i + 2 == end) mac_uniform(lo, hi, a[i], b[q - i], a[i + 1], b[q - i - 1]);
            else if (i + 1 == end) mac_uniform(lo, hi, a[i], b[q - i]);
        } else {
#pragma unroll
            for (; i < end; i++) lo = (uint32_t)lo + a[i] * b[q - i];
        }
        out[q] = (uint32_t)lo;
        lo = (lo >> 32) | ((uint64_t)hi << 32);
    }
}

// floor(k g / 2^256), NC words.  The products below column 6 add less than
// (NG + 1) 2^224: unless word 7 is within that of its end, they change
// nothing above it; else (7 of 2^32 scalars) the whole product is taken.
template <int NG, int NC>
__device__ __forceinline__ void mul_high(const uint32_t* k, const uint32_t* g, uint32_t* out) {
    uint32_t w[8 + NG];
    mul_columns<8, NG, 6, 7 + NC>(k, g, w);
    if (w[7] >= 0u - (uint32_t)(NG + 2)) mul_wide<8, NG>(k, g, w);
#pragma unroll
    for (int i = 0; i < NC; i++) out[i] = w[8 + i];
}

// a = |a| of a two's complement value; returns whether it was negative
__device__ __forceinline__ bool abs128(uint32_t a[4]) {
    const uint32_t s = (uint32_t)((int32_t)a[3] >> 31);
    unsigned br = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) a[i] = __builtin_subc(a[i] ^ s, s, br, &br);
    return s != 0;
}

// Only the low 128 bits of k1 and k2 are formed: both are below 2^127 in
// magnitude, so bit 127 is their sign.  With whole products and k1 folded
// mod r this was two thirds of the decomposition's instructions.
__device__ inline GlvSplit glv_split(const uint32_t kin[8]) {
    uint32_t k[8];
#pragma unroll
    for (int i = 0; i < 8; i++) k[i] = kin[i];
#pragma unroll 1
    for (int it = 0; it < 6 && geq_r(k); it++) {
        uint32_t rr[8];
#pragma unroll
        for (int i = 0; i < 8; i++) rr[i] = r_limb(i);
        sub_n<8>(k, rr);
    }
    const uint32_t g1[5] = {0x391eb18du, 0x7a7bd9d4u, 0xa773d2cfu, 0x4ccef014u, 0x2u};
    const uint32_t g2[3] = {0xc7e0b3d7u, 0xd91d232eu, 0x2u};
    const uint32_t a1[2] = {0x94d213e3u, 0x89d32568u};  // also b2
    const uint32_t a2[4] = {0x1221250bu, 0x0be4e154u, 0xeeb859fdu, 0x6f4d8248u};
    const uint32_t mb1[4] = {0x7d4f1128u, 0x8211bbebu, 0xeeb859fcu, 0x6f4d8248u};
    uint32_t c1[4], c2[2];
    mul_high<5, 4>(k, g1, c1);
    mul_high<3, 2>(k, g2, c2);

    GlvSplit s;
    uint32_t t[4], u[4];
    // k1 = k - c1 a2 - c2 a1
    mul_columns<4, 4, 0, 3>(c1, a2, t);
    mul_columns<2, 2, 0, 3>(c2, a1, u);
#pragma unroll
    for (int i = 0; i < 4; i++) s.k1[i] = k[i];
    sub_n<4>(s.k1, t);
    sub_n<4>(s.k1, u);
    s.neg1 = abs128(s.k1);
    // k2 = c2 (-b1) - c1 b2
    mul_columns<2, 4, 0, 3>(c2, mb1, s.k2);
    mul_columns<4, 2, 0, 3>(c1, a1, u);
    sub_n<4>(s.k2, u);
    s.neg2 = abs128(s.k2);
    return s;
}

// Digit word layout (one per window per half-scalar):
//   0xFFFF when d == 0 (no bucket), else the sort key of bucket |d| - 1
//   (key_encode: bit 7 is free), with bit 7 set if the point is subtracted
//   (digit sign xor GLV sign); never set beside the largest key, 0xFF7F
#define ZK_KEY_NONE 0xFFFFu
#define ZK_SIGN 0x80u

}  // namespace zk
