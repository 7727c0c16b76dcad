// XYZZ point arithmetic by teams of lanes: one lane per coordinate, so an
// addition is four product levels deep instead of fourteen products long.
//
// Why: the bucket merge, the bucket reduction and the window combine are
// chains of dependent additions with too few of them to fill the chip.  One
// lane per addition issues its ~3,300 instructions one after another -- 7.5 us
// per addition whether or not the wave's other lanes have work.  A team
// computes the independent products of one level in different lanes: ~1,200
// instructions, 2.6 us per addition (MI355X, one wave per SIMD).  In lanes spent
// it costs 16 products where one lane needs 14, so it also holds its own where
// the chip is full.
//
//   TeamG1<F>: 4 lanes, lane j holds coordinate j of (X, Y, ZZ, ZZZ).
//   TeamG2:    8 lanes, lane 4k + j holds component k of coordinate j (the
//              stored form's two halves); a product takes the partner lane's
//              components and merges the reduction: c0 = a0 b0 + a1 (10p - b1),
//              c1 = a0 b1 + a1 b0.
//
// Lanes of a team always run together: the callers' branches are uniform per
// team (the cross-lane moves read the team's other lanes).
//
// Bounds, in multiples of p: points in and out X < 6.5p, Y < 4p (G2: 3.5p),
// ZZ, ZZZ < 2p, limbs normalised; a product of operands a, b is below
// ab/169 + 1 (G1), (ab + 10a)/169 + 1 (G2, b < 10), and 2^-29 (Arith::q_m):
// below 1.5 unless noted.
#pragma once
#include "curve29.hpp"
#include "curve_g2.hpp"

namespace zk {

// x from lane CTRL[j] of the quad (dpp quad_perm), per word.  The empty asm
// keeps the move an instruction of its own: folded into a subtraction as the
// subtrahend it becomes v_subrev_u32_dpp, which returns the difference with
// the wrong sign on gfx950 (a - quad_perm(a) came out negated in a four-line
// kernel built with ROCm 7.2).
template <int CTRL>
__device__ __forceinline__ uint32_t quad_perm1(uint32_t a) {
    uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)a, CTRL, 0xf, 0xf, true);
    asm("" : "+v"(r));
    return r;
}
template <int CTRL>
__device__ __forceinline__ Fq quad_perm(const Fq& a) {
    Fq r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.v[i] = quad_perm1<CTRL>(a.v[i]);
    return r;
}
constexpr int qp(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }

// the word of lane ^ 4 (dpp row shifts by four lanes, each into its own banks)
__device__ __forceinline__ uint32_t swap4(uint32_t a) {
    const int up = __builtin_amdgcn_update_dpp(0, (int)a, 0x104, 0xf, 0x5, false);  // row_shl:4
    uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(up, (int)a, 0x114, 0xf, 0xa, false);  // row_shr:4
    asm("" : "+v"(r));
    return r;
}
__device__ __forceinline__ Fq swap4(const Fq& a) {
    Fq r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.v[i] = swap4(a.v[i]);
    return r;
}

// the field element of a lane and its product, per curve
template <class F>
struct TeamFieldG1 {
    using A = Arith<F>;
    using Field = F;
    static constexpr uint32_t kLanes = 4;
    static constexpr uint64_t kPtBytes = kBucketBytes;
    static __device__ __forceinline__ Fq mul(const Fq& a, const Fq& b) { return A::fq_mul(a, b); }
    // all of the team's copies of a component test
    static __device__ __forceinline__ uint32_t both(uint32_t z) { return z; }
    static __device__ __forceinline__ uint64_t word0(uint64_t i, uint32_t t) { return i * 36 + t * 9; }
};

struct TeamFieldG2 {
    using A = Arith<Bn254Fp>;
    using Field = Bn254Fp;
    static constexpr uint32_t kLanes = 8;
    static constexpr uint64_t kPtBytes = 2 * kBucketBytes;
    static __device__ __forceinline__ Fq mul(const Fq& a, const Fq& b) {
        const Fq ao = swap4(a), bo = swap4(b);
        const bool hi = (__lane_id() & 4u) != 0;
        Fq x, y, z;
#pragma unroll
        for (int i = 0; i < 9; i++) {
            x.v[i] = hi ? ao.v[i] : a.v[i];
            y.v[i] = hi ? a.v[i] : ao.v[i];
            z.v[i] = hi ? bo.v[i] : A::template q_kpr<10>(i) - bo.v[i];
        }
        // component 0: a0 b0 + a1 (10p - b1); component 1: a0 b1 + a1 b0
        return A::fq_mul_add(x, b, y, z);
    }
    static __device__ __forceinline__ uint32_t both(uint32_t z) { return z & swap4(z); }
    static __device__ __forceinline__ uint64_t word0(uint64_t i, uint32_t t) { return i * 72 + t * 9; }
};

template <class TF>
struct Team {
    using A = typename TF::A;
    using Field = typename TF::Field;
    using Pt = Fq;  // this lane's coordinate (component)
    static constexpr uint32_t kLanes = TF::kLanes;
    static constexpr uint32_t kPerWave = 64 / kLanes;
    static constexpr uint64_t kPtBytes = TF::kPtBytes;

    static __device__ __forceinline__ uint32_t lane() { return __lane_id() & (kLanes - 1); }
    static __device__ __forceinline__ Pt identity() { return fq_zero(); }
    static __device__ __forceinline__ Pt select(bool c, const Pt& a, const Pt& b) { return fq_select(c, a, b); }

    // stored points (the limbs of X, Y, ZZ, ZZZ, 9 words each): 36 consecutive
    // bytes per lane, 144 (288) per team
    static __device__ __forceinline__ Pt load(const uint4* b, uint64_t i) {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(b) + TF::word0(i, lane());
        Pt r;
#pragma unroll
        for (int k = 0; k < 9; k++) r.v[k] = p[k];
        return r;
    }
    static __device__ __forceinline__ void store(uint4* b, uint64_t i, const Pt& a) {
        uint32_t* p = reinterpret_cast<uint32_t*>(b) + TF::word0(i, lane());
#pragma unroll
        for (int k = 0; k < 9; k++) p[k] = a.v[k];
    }
    // host form: the coordinates as canonical 2^256 Montgomery integers, 32 B
    // per lane (G2: the c0 record, then the c1 record)
    static __device__ __forceinline__ void store_host(uint4* b, uint64_t i, const Pt& a) {
        const Fp f = A::fq_to_fp(a);
        uint4* o = b + (i * kLanes + lane()) * 2;
        o[0] = make_uint4(f.v[0], f.v[1], f.v[2], f.v[3]);
        o[1] = make_uint4(f.v[4], f.v[5], f.v[6], f.v[7]);
    }
    // the point of the team s teams away (xor), s a power of two below kPerWave
    static __device__ __forceinline__ Pt xor_team(const Pt& a, uint32_t s) {
        Pt r;
#pragma unroll
        for (int k = 0; k < 9; k++) r.v[k] = (uint32_t)__shfl_xor((int)a.v[k], (int)(s * kLanes));
        return r;
    }
    // value < 2p == 0 mod p, agreed by the coordinate's lanes
    static __device__ __forceinline__ uint32_t zero(const Fq& a) {
        return TF::both(A::fq_is_zero2(a) ? 1u : 0u);
    }
    // the point is the identity (ZZ = 0), known to every lane
    static __device__ __forceinline__ uint32_t is_id(const Pt& a) {
        return quad_perm1<qp(2, 2, 2, 2)>(zero(a));
    }

    // 2 a (dbl-2008-s-1, a = 0): three product levels.  The identity stays the
    // identity.  Out: X < 4.5p, Y < 3.5p, ZZ, ZZZ < 1.5p.
    static __device__ __forceinline__ Pt dbl(const Pt& a) {
        const uint32_t j = lane() & 3u;
        const Fq U = A::fq_add(a, a);                    // lane 1: 2Y < 8p
        const Fq t = fq_select(j == 1, U, a);
        const Fq p1 = TF::mul(t, t);                     // X^2 < 1.7p | V = U^2 < 1.8p | - | -
        const Fq xx = quad_perm<qp(0, 0, 0, 0)>(p1);
        const Fq M = A::fq_add(A::fq_add(xx, xx), xx);   // < 5.1p
        const Fq V = quad_perm<qp(1, 1, 1, 1)>(p1);
        const Fq a2 = fq_select(j == 3, M, t);
        const Fq b2 = fq_select(j == 3, M, V);
        const Fq p2 = TF::mul(a2, b2);                   // S = X V | W = U V | ZZ3 | M^2
        const Fq S = quad_perm<qp(0, 0, 0, 0)>(p2);
        const Fq W = quad_perm<qp(1, 1, 1, 1)>(p2);
        const Fq X3 = A::template fq_sub<3>(quad_perm<qp(3, 3, 3, 3)>(p2), A::fq_add(S, S));  // < 4.5p
        const Fq a3 = fq_select(j == 0, M, W);
        const Fq b3 = fq_select(j == 0, A::template fq_sub<5>(S, X3), a);
        const Fq p3 = TF::mul(a3, b3);                   // M (S - X3) | W Y | - | ZZZ3
        const Fq Y3 = A::template fq_sub<2>(quad_perm<qp(0, 0, 0, 0)>(p3), p3);
        return fq_select(j == 0, X3, fq_select(j == 1, Y3, fq_select(j == 2, p2, p3)));
    }

    // a += b (add-2008-s), every case: identities, doubling, cancellation
    // (P = 0 gives ZZ3 = 0, the identity).  Out: X < 6.5p, Y < 3.5p, ZZ, ZZZ < 1.5p.
    static __device__ __forceinline__ void add(Pt& a, const Pt& b) {
        const uint32_t j = lane() & 3u;
        const Fq p1 = TF::mul(a, quad_perm<qp(2, 3, 0, 1)>(b));           // U1 | S1 | U2 | S2
        // U1 - U2 | S1 - S2 | P = U2 - U1 | R = S2 - S1, < 3.5p
        const Fq D = A::template fq_sub<2>(p1, quad_perm<qp(2, 3, 0, 1)>(p1));
        const Fq p2 = TF::mul(fq_select(j < 2, D, a), fq_select(j < 2, D, b));  // PP | RR | ZZ1 ZZ2 | ZZZ1 ZZZ2
        const Fq PP = quad_perm<qp(0, 0, 0, 0)>(p2);
        const Fq a3 = fq_select(j < 2, p1, fq_select(j == 2, p2, quad_perm<qp(2, 2, 2, 2)>(D)));
        const Fq p3 = TF::mul(a3, PP);                                     // Q = U1 PP | - | ZZ3 | PPP
        const Fq Q = quad_perm<qp(0, 0, 0, 0)>(p3);
        const Fq PPP = quad_perm<qp(3, 3, 3, 3)>(p3);
        Fq T;  // 2Q + PPP < 4.5p, limbs sums of three normalised limbs
#pragma unroll
        for (int i = 0; i < 9; i++) T.v[i] = Q.v[i] + Q.v[i] + PPP.v[i];
        const Fq X3 = A::template fq_sub<5>(quad_perm<qp(1, 1, 1, 1)>(p2), T);  // < 6.5p
        const Fq a4 = fq_select(j == 0, quad_perm<qp(3, 3, 3, 3)>(D), PPP);
        const Fq b4 = fq_select(j == 0, A::template fq_sub<7>(Q, X3), fq_select(j == 1, p1, p2));
        const Fq p4 = TF::mul(a4, b4);                                     // R (Q - X3) | S1 PPP | - | ZZZ3
        const Fq Y3 = A::template fq_sub<2>(quad_perm<qp(0, 0, 0, 0)>(p4), p4);
        Pt r = fq_select(j == 0, X3, fq_select(j == 1, Y3, fq_select(j == 2, p3, p4)));
        // PP = 0, RR = 0 or ZZ1 ZZ2 = 0 anywhere in the wave: the exceptions
        const uint32_t z = zero(p2) & (uint32_t)(j != 3);
        if (__any((int)z)) {
            const uint32_t aid = is_id(a), bid = is_id(b);
            const uint32_t same = quad_perm1<qp(0, 0, 0, 0)>(z) & quad_perm1<qp(1, 1, 1, 1)>(z) & (aid ^ 1u) & (bid ^ 1u);
            if (__any((int)same)) r = fq_select(same != 0, dbl(a), r);
            r = fq_select(aid != 0, b, r);
            r = fq_select(bid != 0, a, r);
        }
        a = r;
    }
};

template <class F>
using TeamG1 = Team<TeamFieldG1<F>>;
using TeamG2 = Team<TeamFieldG2>;

}  // namespace zk
