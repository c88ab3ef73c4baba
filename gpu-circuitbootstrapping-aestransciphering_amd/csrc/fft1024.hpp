// fft1024.hpp -- negacyclic FP64 FFT for N = 2048 (M = 1024 complex points)
// distributed over the four wavefronts of a workgroup.
//
// Decimation in time by 4: wave r owns the folded points z_j, j = 4m + r
// (m = 64a + b: lane b, slot a < 4), i.e. coefficients 4m + r (real part) and
// 4m + r + 1024 (imaginary part).  Each wave runs an LDS-transposed radix-4
// 256-point FFT on its subsequence (twisted by (w^4)^m, w = exp(i pi / N)),
// multiplies by T_r[k] = w^r W1024^(r k), and one cross-wave radix-4 step gives
// wave q the frequencies Z[k + 256 q].  Frequency layout of a transformed
// polynomial: [q][slot s < 4][lane] with k = k0 + 4e + 16p + 64s for lane
// 16 k0 + 4e + p.  The inverse runs the steps backwards and returns
// 1024 x the folded pairs in the same coefficient ownership, so a polynomial
// never leaves the wave that decomposes it.
#pragma once
#include "device_common.hpp"

namespace tfhe {

constexpr int F256_LDS_CPLX = 320;  // per-wave transpose buffer (bank-staggered rows)

// The transform is written once for a complex type C: cplx (FP64, every form of the
// bootstraps) or cplxf (FP32, the split-precision product); tables hold C values.
template <class C>
struct FFT1024TablesT {
    const C* p1t;  // [4 k0][64 b]  (w^4)^b * W256^(b k0)
    const C* p2;   // [4 e][64 L]   W64^((L mod 16) e)
    const C* p3;   // [4 p][64 L]   W16^((L mod 4) p)
    const C* tr;   // [4 r][4 s][64 lane]  w^r W1024^(r k(lane, s))
    const C* rot;  // [2N] w^j: frequency k (wave q, slot s, lane) is the polynomial at w^(1 - 4k),
                   // k = (lane >> 4) + 4 ((lane >> 2) & 3) + 16 (lane & 3) + 64 s + 256 q
    const C* pw;   // [10][16 L = 4 k0 + e] of fft_rows.hpp's fused form: with v = w^4 W256^(k0 + 4 e):
                   // v^4, v^8, then v_p, v_p^2 for v_p = v W16^p, p < 4
};
using FFT1024Tables = FFT1024TablesT<cplx>;
using FFT1024TablesF = FFT1024TablesT<cplxf>;

// (w^4)^(64 a) = exp(i pi a / 8), a < 4
template <class C = cplx>
__device__ __forceinline__ C twist4_const(int a) {
    using S = decltype(C{}.re);
    constexpr double K[4][2] = {{1.0, 0.0},
                                {0.92387953251128674, 0.38268343236508978},
                                {0.70710678118654757, 0.70710678118654746},
                                {0.38268343236508984, 0.92387953251128674}};
    return {(S)K[a][0], (S)K[a][1]};
}

template <bool INV, class C>
__device__ __forceinline__ void dft4(C (&x)[4]) {
    C a0 = cadd(x[0], x[2]), a1 = csub(x[0], x[2]);
    C b0 = cadd(x[1], x[3]), b1 = mul_mi<INV>(csub(x[1], x[3]));
    x[0] = cadd(a0, b0);
    x[2] = csub(a0, b0);
    x[1] = cadd(a1, b1);
    x[3] = csub(a1, b1);
}

// x + w y and 2 x - s
__device__ __forceinline__ cplx cfma(cplx x, cplx w, cplx y) {
    return {fma(-w.im, y.im, fma(w.re, y.re, x.re)), fma(w.im, y.re, fma(w.re, y.im, x.im))};
}
__device__ __forceinline__ cplx twice_less(cplx x, cplx s) { return {fma(2.0, x.re, -s.re), fma(2.0, x.im, -s.im)}; }
// radix-4 of x[j] w^j, w1 = w, w2 = w^2
template <bool INV>
__device__ __forceinline__ void dft4_pw(cplx (&x)[4], cplx w1, cplx w2) {
    const cplx e = cfma(x[0], w2, x[2]), f = twice_less(x[0], e);
    const cplx g = cfma(x[1], w2, x[3]), h = twice_less(x[1], g);
    x[0] = cfma(e, w1, g);
    x[2] = twice_less(e, x[0]);
    x[1] = cfma(f, mul_mi<INV>(w1), h);
    x[3] = twice_less(f, x[1]);
}
__device__ __forceinline__ cplx cconj(cplx a) { return {a.re, -a.im}; }

// exp(i pi j / 32) for the constants of the first two steps
__device__ __forceinline__ cplx pw_const(int j) {
    constexpr double C[17] = {1.0, 0.99518472667219693, 0.98078528040323043, 0.95694033573220882, 0.92387953251128674,
                              0.88192126434835505, 0.83146961230254524, 0.77301045336273699, 0.70710678118654757,
                              0.63439328416364549, 0.55557023301960229, 0.47139673682599764, 0.38268343236508978,
                              0.29028467725446233, 0.19509032201612828, 0.098017140329560604, 0.0};
    const int a = j < 0 ? -j : j, im = a <= 16 ? 16 - a : a - 16;  // |j| <= 32
    const double c = a <= 16 ? C[a] : -C[32 - a], s = C[im];
    return {c, j < 0 ? -s : s};
}

// The first transpose of the forward 256-point step (and the last of the inverse, its own
// inverse): slot c of lane 16 q + d takes slot q of lane 16 c + d, a 4 x 4 transpose of
// (slot, 16-lane row) done in registers by gfx950's row swaps: v_permlane32_swap exchanges
// rows 2, 3 of one register with rows 0, 1 of another, v_permlane16_swap rows 1, 3 with
// rows 0, 2.  Slots (0, 2), (1, 3) through the first, then (0, 1), (2, 3) through the second.
template <class C>
__device__ __forceinline__ void row_transpose4(C (&x)[4]) {
    constexpr int W = (int)(sizeof(C) / 4);  // dwords per value
    uint32_t d[4][W];
#pragma unroll
    for (int s = 0; s < 4; ++s) __builtin_memcpy(d[s], &x[s], sizeof(C));
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const auto a = __builtin_amdgcn_permlane32_swap(d[0][w], d[2][w], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(d[1][w], d[3][w], false, false);
        const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
        const auto e = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
        d[0][w] = c[0];
        d[1][w] = c[1];
        d[2][w] = e[0];
        d[3][w] = e[1];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) __builtin_memcpy(&x[s], d[s], sizeof(C));
}
__device__ __forceinline__ int f256_a2(int k0, int e, int d) { return k0 * 80 + e * 20 + d; }
__device__ __forceinline__ int f256_a3(int k0, int e, int p, int h) { return k0 * 80 + e * 20 + p * 5 + h; }

// twiddles of the 256-point step: p1(k), p2(e), p3(p) of one lane, read from the tables ...
template <class C>
struct Tw256 {
    const C *p1t, *p2t, *p3t;  // at this lane
    __device__ __forceinline__ Tw256(const FFT1024TablesT<C>& T, int lane)
        : p1t(T.p1t + lane), p2t(T.p2 + lane), p3t(T.p3 + lane) {}
    __device__ __forceinline__ C p1(int k) const { return p1t[k * 64]; }
    __device__ __forceinline__ C p2(int e) const { return p2t[e * 64]; }
    __device__ __forceinline__ C p3(int p) const { return p3t[p * 64]; }
};
// ... or held in registers: they are the same for every transform a lane runs
struct Tw256Regs {
    cplx a[4], b[3], c[3];
    __device__ __forceinline__ Tw256Regs(const FFT1024Tables& T, int lane) {
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = T.p1t[k * 64 + lane];
#pragma unroll
        for (int e = 1; e < 4; ++e) {
            b[e - 1] = T.p2[e * 64 + lane];
            c[e - 1] = T.p3[e * 64 + lane];
        }
    }
    __device__ __forceinline__ cplx p1(int k) const { return a[k]; }
    __device__ __forceinline__ cplx p2(int e) const { return b[e - 1]; }
    __device__ __forceinline__ cplx p3(int p) const { return c[p - 1]; }
};

// forward 256-point: x = untwisted folded points (lane b, slot a -> point 64a + b)
template <class C, class Tw>
__device__ __forceinline__ void fft256_fwd(C (&x)[4], C* lds, const Tw& T, int lane) {
#pragma unroll
    for (int a = 1; a < 4; ++a) x[a] = cmul(x[a], twist4_const<C>(a));
    dft4<false>(x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = cmul(x[k], T.p1(k));
    row_transpose4(x);
    const int k0 = lane >> 4, d = lane & 15;
    dft4<false>(x);
#pragma unroll
    for (int e = 1; e < 4; ++e) x[e] = cmul(x[e], T.p2(e));
#pragma unroll
    for (int e = 0; e < 4; ++e) lds[f256_a2(k0, e, d)] = x[e];
    wave_sync();
    const int e = (lane >> 2) & 3, h = lane & 3;
#pragma unroll
    for (int g = 0; g < 4; ++g) x[g] = lds[f256_a2(k0, e, 4 * g + h)];
    wave_sync();
    dft4<false>(x);
#pragma unroll
    for (int p = 1; p < 4; ++p) x[p] = cmul(x[p], T.p3(p));
#pragma unroll
    for (int p = 0; p < 4; ++p) lds[f256_a3(k0, e, p, h)] = x[p];
    wave_sync();
    const int pp = lane & 3;
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) x[hh] = lds[f256_a3(k0, e, pp, hh)];
    wave_sync();
    dft4<false>(x);
}

// inverse 256-point: frequency layout in, 256 x folded points out
template <class C, class Tw>
__device__ __forceinline__ void fft256_inv(C (&x)[4], C* lds, const Tw& T, int lane) {
    dft4<true>(x);
    const int k0 = lane >> 4, e = (lane >> 2) & 3, low = lane & 3;
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) lds[f256_a3(k0, e, low, hh)] = x[hh];
    wave_sync();
#pragma unroll
    for (int p = 0; p < 4; ++p) x[p] = lds[f256_a3(k0, e, p, low)];
    wave_sync();
#pragma unroll
    for (int p = 1; p < 4; ++p) x[p] = cmulc(x[p], T.p3(p));
    dft4<true>(x);
#pragma unroll
    for (int g = 0; g < 4; ++g) lds[f256_a2(k0, e, 4 * g + low)] = x[g];
    wave_sync();
    const int d = lane & 15;
#pragma unroll
    for (int ee = 0; ee < 4; ++ee) x[ee] = lds[f256_a2(k0, ee, d)];
    wave_sync();
#pragma unroll
    for (int ee = 1; ee < 4; ++ee) x[ee] = cmulc(x[ee], T.p2(ee));
    dft4<true>(x);
    row_transpose4(x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = cmulc(x[k], T.p1(k));
    dft4<true>(x);
#pragma unroll
    for (int a = 1; a < 4; ++a) x[a] = cmulc(x[a], twist4_const<C>(a));
}

// The 256-point step with the twiddles fused into the butterflies (for products that are rounded
// to integers, whose words do not depend on the order of the FP64 operations): point
// b = 64 a + 16 c + d carries v0^b, v0 = w^4, and k = k0 + 4 e + 16 p + 64 s; over c powers of
// (v0 W256^k0)^16, over g and h (d = 4 g + h) powers of v^4 and v W16^p, v = v0 W256^(k0 + 4 e).
struct Pw256Regs {  // each pair: the factor and its square at this lane
    cplx w[6];
    __device__ __forceinline__ Pw256Regs(const cplx* t, int lane) {
#pragma unroll
        for (int k = 0; k < 6; ++k) w[k] = t[k * 64 + lane];
    }
};
__device__ __forceinline__ void fft256_fwd_pw(cplx (&x)[4], cplx* lds, const Pw256Regs& T, int lane) {
    dft4_pw<false>(x, pw_const(4), pw_const(8));
    row_transpose4(x);
    const int k0 = lane >> 4, d = lane & 15, e = (lane >> 2) & 3, low = lane & 3;
    dft4_pw<false>(x, T.w[0], T.w[1]);
#pragma unroll
    for (int q = 0; q < 4; ++q) lds[f256_a2(k0, q, d)] = x[q];
    wave_sync();
#pragma unroll
    for (int g = 0; g < 4; ++g) x[g] = lds[f256_a2(k0, e, 4 * g + low)];
    wave_sync();
    dft4_pw<false>(x, T.w[2], T.w[3]);
#pragma unroll
    for (int p = 0; p < 4; ++p) lds[f256_a3(k0, e, p, low)] = x[p];
    wave_sync();
#pragma unroll
    for (int h = 0; h < 4; ++h) x[h] = lds[f256_a3(k0, e, low, h)];
    wave_sync();
    dft4_pw<false>(x, T.w[4], T.w[5]);
}
template <class Tw>
__device__ __forceinline__ void fft256_inv_pw(cplx (&x)[4], cplx* lds, const Tw& T, int lane) {
    dft4<true>(x);
    const int k0 = lane >> 4, e = (lane >> 2) & 3, low = lane & 3, d = lane & 15;
#pragma unroll
    for (int h = 0; h < 4; ++h) lds[f256_a3(k0, e, low, h)] = x[h];
    wave_sync();
#pragma unroll
    for (int p = 0; p < 4; ++p) x[p] = lds[f256_a3(k0, e, p, low)];
    wave_sync();
    dft4_pw<true>(x, cconj(T.p3(1)), cconj(T.p3(2)));
#pragma unroll
    for (int g = 0; g < 4; ++g) lds[f256_a2(k0, e, 4 * g + low)] = x[g];
    wave_sync();
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = lds[f256_a2(k0, q, d)];
    wave_sync();
    dft4_pw<true>(x, cconj(T.p2(1)), cconj(T.p2(2)));
    row_transpose4(x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = cmulc(x[k], T.p1(k));
    dft4<true>(x);
#pragma unroll
    for (int a = 1; a < 4; ++a) x[a] = cmulc(x[a], twist4_const<cplx>(a));
}

// Cross-wave step of the FFT1024 (wave w holds frequencies 256 w ..): forward and
// inverse, with the cross twiddles trw taken from registers; the radix-4 output of wave w
// is selected on w (uniform branches).  xbuf: 1024 C of LDS shared by the four waves.  (The
// bootstraps run fft_rows.hpp, which computes each radix-4 once.)
template <class C>
__device__ __forceinline__ void f1024_fwd(C (&x)[4], C* lds, C* xbuf, const FFT1024TablesT<C>& T,
                                          const C (&trw)[4], int w, int lane) {
    fft256_fwd(x, lds, Tw256<C>(T, lane), lane);
#pragma unroll
    for (int s = 0; s < 4; ++s) xbuf[(w * 4 + s) * 64 + lane] = cmul(x[s], trw[s]);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        C y0 = xbuf[(0 * 4 + s) * 64 + lane], y1 = xbuf[(1 * 4 + s) * 64 + lane];
        C y2 = xbuf[(2 * 4 + s) * 64 + lane], y3 = xbuf[(3 * 4 + s) * 64 + lane];
        C s02 = cadd(y0, y2), d02 = csub(y0, y2), s13 = cadd(y1, y3), d13 = mul_mi<false>(csub(y1, y3));
        x[s] = (w == 0) ? cadd(s02, s13) : (w == 1) ? cadd(d02, d13) : (w == 2) ? csub(s02, s13) : csub(d02, d13);
    }
}

template <class C>
__device__ __forceinline__ void f1024_inv(C (&x)[4], C* lds, C* xbuf, const FFT1024TablesT<C>& T,
                                          const C (&trw)[4], int w, int lane) {
#pragma unroll
    for (int s = 0; s < 4; ++s) xbuf[(w * 4 + s) * 64 + lane] = x[s];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        C z0 = xbuf[(0 * 4 + s) * 64 + lane], z1 = xbuf[(1 * 4 + s) * 64 + lane];
        C z2 = xbuf[(2 * 4 + s) * 64 + lane], z3 = xbuf[(3 * 4 + s) * 64 + lane];
        C s02 = cadd(z0, z2), d02 = csub(z0, z2), s13 = cadd(z1, z3), d13 = mul_mi<true>(csub(z1, z3));
        const C y =
            (w == 0) ? cadd(s02, s13) : (w == 1) ? cadd(d02, d13) : (w == 2) ? csub(s02, s13) : csub(d02, d13);
        x[s] = cmulc(y, trw[s]);
    }
    fft256_inv(x, lds, Tw256<C>(T, lane), lane);
}

template <class C>
__device__ __forceinline__ void load_trw(const FFT1024TablesT<C>& Tg, int w, int lane, C (&trw)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) trw[s] = Tg.tr[(w * 4 + s) * 64 + lane];
}

// coefficient owned by (wave w, lane, slot a): 4 (64 a + lane) + w; slot a + 4 is +1024
__device__ __forceinline__ int own_coeff(int w, int lane, int a) { return 4 * (64 * a + lane) + w; }

// round(x * scale) mod 2^64 through two FP64 limbs is done by the callers;
// exact int64 of a rounded double with |x| < 2^52.
__device__ __forceinline__ int64_t round_i64(double x, double scale, double magic = ROUND_MAGIC) {
    const double y = fma(x, scale, magic);
    return __double_as_longlong(y) - 0x4338000000000000ll;
}

}  // namespace tfhe
