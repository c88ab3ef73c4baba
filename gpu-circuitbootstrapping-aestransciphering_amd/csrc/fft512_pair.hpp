// fft512_pair.hpp -- two negacyclic N = 1024 transforms (M = 512 complex points) per
// wavefront, one per half: lanes 32 u .. 32 u + 31 hold polynomial u, 16 points per lane.
//
// The transform evaluates z(x) at the roots of x^512 = i by splitting x^m - c into
// x^(m/2) -+ t, t^2 = c (the twist needs no pass of its own): nine levels of butterflies
// lo + t hi, lo - t hi, six FMAs each.  Point 32 a + d starts in slot a of lane d.  Levels
// 1-4 split on the slot's bits with compile-time t; one LDS transpose then gives lane
// (node n, d0) the 16 points d = 2 g + d0 of node n; levels 5-8 split on g's bits, and level
// 9 on d0 after a register swap of 16-lane rows.  A t that belongs to a minus child is i
// times its sibling's, so a lane reads 16 twiddles for its 72 butterflies.  Against one
// transform per wave (8 points per lane, radix 8 x 3) this halves the LDS traffic per
// transform and leaves one LDS round trip where two transforms had four.
//
// Bits b1 .. b9 (1 = the minus child) name a root: x = w^e, w = exp(i pi / 1024),
// e = 1 + 4 b1 + 8 b2 + 16 b3 + 32 b4 + 64 b5 + 128 b6 + 256 b7 + 512 b8 + 1024 b9.
// Frequency order of keys and products: [p = 4 b5 + 2 b6 + b7][lane = n + 16 b8 + 32 b9],
// n = 8 b1 + 4 b2 + 2 b3 + b4.
#pragma once
#include "device_common.hpp"

namespace tfhe {

constexpr int PAIR_LDS_CPLX = 1024;  // one wave's transpose: 2 halves x 16 nodes x 32 points

// LDS tables: levels 5, 6, 7 [b5], 8 [b5 b6] at node n: [8][16], then level 9 [p][n + 16 b8]
constexpr int PAIR_TABLE_CPLX = 8 * 16 + 8 * 32;

__host__ __device__ inline uint32_t rev_bits(uint32_t v, int bits) {
    uint32_t r = 0;
    for (int k = 0; k < bits; ++k) r |= ((v >> k) & 1u) << (bits - 1 - k);
    return r;
}
// position [p][lane] of frequency k of fft512_fwd (the value at w^(1 - 4k)) in the pair order
__host__ __device__ inline uint32_t pair_pos(uint32_t k) {
    const uint32_t K = (512u - k) & 511u;  // (e - 1) / 4
    return rev_bits((K >> 4) & 7, 3) * 64 + rev_bits(K & 15, 4) + 16 * ((K >> 7) & 1) + 32 * (K >> 8);
}

// (p, q) = (lo + s hi, lo - s hi) with s = t, or i t
template <bool I>
__device__ __forceinline__ void pair_bf(cplx& lo, cplx& hi, cplx t) {
    cplx p;
    if constexpr (I) {
        p = {fma(-t.im, hi.re, fma(-t.re, hi.im, lo.re)), fma(-t.im, hi.im, fma(t.re, hi.re, lo.im))};
    } else {
        p = {fma(-t.im, hi.im, fma(t.re, hi.re, lo.re)), fma(t.im, hi.re, fma(t.re, hi.im, lo.im))};
    }
    hi = {fma(2.0, lo.re, -p.re), fma(2.0, lo.im, -p.im)};
    lo = p;
}
// the inverse, times 2: (lo, hi) = (p + q, (p - q) conj(s))
template <bool I>
__device__ __forceinline__ void pair_ibf(cplx& p, cplx& q, cplx t) {
    const cplx d = csub(p, q);
    p = cadd(p, q);
    if constexpr (I) q = {fma(d.im, t.re, -(d.re * t.im)), -fma(d.re, t.re, d.im * t.im)};
    else q = {fma(d.re, t.re, d.im * t.im), fma(d.im, t.re, -(d.re * t.im))};
}

// exp(i pi j / 32), j = 1, 5, 9, 13 (level 4), 2, 10 (level 3), 4 (level 2), 8 (level 1)
__device__ __forceinline__ cplx pair_const(int j) {
    constexpr double C[14][2] = {{1.0, 0.0},
                                 {0.99518472667219693, 0.098017140329560604},
                                 {0.98078528040323043, 0.19509032201612825},
                                 {0.0, 0.0},
                                 {0.92387953251128674, 0.38268343236508978},
                                 {0.88192126434835505, 0.47139673682599764},
                                 {0.0, 0.0},
                                 {0.0, 0.0},
                                 {0.70710678118654757, 0.70710678118654746},
                                 {0.63439328416364549, 0.77301045336273699},
                                 {0.55557023301960229, 0.83146961230254524},
                                 {0.0, 0.0},
                                 {0.0, 0.0},
                                 {0.29028467725446233, 0.95694033573220882}};
    return {C[j][0], C[j][1]};
}

// level L = 1..4 on slot bit 4 - L, INV or forward; the twiddle of a butterfly whose node is
// (b1 .. b(L-1)) = the slot's higher bits
template <int L, bool INV>
__device__ __forceinline__ void pair_slot_level(cplx (&x)[16]) {
    constexpr int H = 16 >> L;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        if (s & H) continue;
        // angle pi / 2^(L+1) + pi (b1 / 2^(L-1) + .. + b(L-2) / 4), times i for b(L-1)
        int j = 32 >> (L + 1);
#pragma unroll
        for (int l = 1; l <= L - 2; ++l)
            if (s & (16 >> l)) j += 32 >> (L - l);
        const bool I = L > 1 && (s & (2 * H));
        if (I) {
            if constexpr (INV) pair_ibf<true>(x[s], x[s + H], pair_const(j));
            else pair_bf<true>(x[s], x[s + H], pair_const(j));
        } else {
            if constexpr (INV) pair_ibf<false>(x[s], x[s + H], pair_const(j));
            else pair_bf<false>(x[s], x[s + H], pair_const(j));
        }
    }
}
// level L = 5..8 on slot bit 8 - L; t: this lane's twiddles of the level, by the higher slot
// bits without the last
template <int L, bool INV>
__device__ __forceinline__ void pair_lane_level(cplx (&x)[16], const cplx* t) {
    constexpr int H = 16 >> (L - 4);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        if (s & H) continue;
        const cplx tw = t[(s / (4 * H)) * 16];
        if (L > 5 && (s & (2 * H))) {
            if constexpr (INV) pair_ibf<true>(x[s], x[s + H], tw);
            else pair_bf<true>(x[s], x[s + H], tw);
        } else {
            if constexpr (INV) pair_ibf<false>(x[s], x[s + H], tw);
            else pair_bf<false>(x[s], x[s + H], tw);
        }
    }
}

// exchanges lane bit 4 (or 5) with the slot bit between a and b
__device__ __forceinline__ void swap_rows16(cplx& a, cplx& b) {
    uint32_t u[4], v[4];
    __builtin_memcpy(u, &a, 16);
    __builtin_memcpy(v, &b, 16);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const auto s = __builtin_amdgcn_permlane16_swap(u[w], v[w], false, false);
        u[w] = s[0];
        v[w] = s[1];
    }
    __builtin_memcpy(&a, u, 16);
    __builtin_memcpy(&b, v, 16);
}
__device__ __forceinline__ void swap_rows32(cplx& a, cplx& b) {
    uint32_t u[4], v[4];
    __builtin_memcpy(u, &a, 16);
    __builtin_memcpy(v, &b, 16);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const auto s = __builtin_amdgcn_permlane32_swap(u[w], v[w], false, false);
        u[w] = s[0];
        v[w] = s[1];
    }
    __builtin_memcpy(&a, u, 16);
    __builtin_memcpy(&b, v, 16);
}

// LDS addresses of the transpose: element (node a, d) at a * 32 + (d ^ (a & 7)), so that
// both sides (fixed a, lanes d; lanes a, fixed d) touch all banks
struct PairAddr {
    cplx* by_node;   // this half; + 32 a + (d ^ (a & 7))
    cplx* by_point;  // this half and node
    int d, n7, d0;
    __device__ __forceinline__ PairAddr(cplx* lds, int lane)
        : by_node(lds + (lane >> 5) * 512), by_point(lds + (lane >> 5) * 512 + (lane & 15) * 32), d(lane & 31),
          n7(lane & 7), d0((lane >> 4) & 1) {}
    __device__ __forceinline__ cplx& node(int a) const { return by_node[(d ^ (a & 7)) + 32 * a]; }
    __device__ __forceinline__ cplx& point(int g) const { return by_point[((2 * (g & 3) + d0) ^ n7) + 8 * (g >> 2)]; }
};

// forward: slot a = point 32 a + d of polynomial u = lane >> 5; out: x[2 p + b9] at lane
// (n, b8) of half u
__device__ __forceinline__ void fft512_pair_fwd(cplx (&x)[16], const PairAddr& A, const cplx* tab, int lane) {
    pair_slot_level<1, false>(x);
    pair_slot_level<2, false>(x);
    pair_slot_level<3, false>(x);
    pair_slot_level<4, false>(x);
#pragma unroll
    for (int a = 0; a < 16; ++a) A.node(a) = x[a];
    wave_sync();
#pragma unroll
    for (int g = 0; g < 16; ++g) x[g] = A.point(g);
    wave_sync();
    const cplx* t = tab + (lane & 15);
    pair_lane_level<5, false>(x, t);
    pair_lane_level<6, false>(x, t + 16);
    pair_lane_level<7, false>(x, t + 32);
    pair_lane_level<8, false>(x, t + 64);
    const cplx* t9 = tab + 128 + (lane & 31);
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        swap_rows16(x[2 * p], x[2 * p + 1]);
        pair_bf<false>(x[2 * p], x[2 * p + 1], t9[32 * p]);
    }
}

// inverse of the same, times 512
__device__ __forceinline__ void fft512_pair_inv(cplx (&x)[16], const PairAddr& A, const cplx* tab, int lane) {
    const cplx* t9 = tab + 128 + (lane & 31);
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        pair_ibf<false>(x[2 * p], x[2 * p + 1], t9[32 * p]);
        swap_rows16(x[2 * p], x[2 * p + 1]);
    }
    const cplx* t = tab + (lane & 15);
    pair_lane_level<8, true>(x, t + 64);
    pair_lane_level<7, true>(x, t + 32);
    pair_lane_level<6, true>(x, t + 16);
    pair_lane_level<5, true>(x, t);
#pragma unroll
    for (int g = 0; g < 16; ++g) A.point(g) = x[g];
    wave_sync();
#pragma unroll
    for (int a = 0; a < 16; ++a) x[a] = A.node(a);
    wave_sync();
    pair_slot_level<4, true>(x);
    pair_slot_level<3, true>(x);
    pair_slot_level<2, true>(x);
    pair_slot_level<1, true>(x);
}

}  // namespace tfhe
