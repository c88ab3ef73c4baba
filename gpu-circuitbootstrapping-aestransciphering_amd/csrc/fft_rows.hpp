// fft_rows.hpp -- the N = 2048 transform of fft1024.hpp for several polynomials at once.
//
// The four waves of an FFT1024 each run one 256-point transform per polynomial and meet in
// a cross-wave radix-4 step.  Here a wave runs FOUR 256-point transforms together (the four
// digit rows of one accumulator polynomial, or the four inverse transforms of the exact
// form): lane group R = lane >> 4 holds transform R, 16 points per lane, so that two of its
// four radix-4 layers need no exchange, the next two meet after one 16 x 16 transpose
// through LDS, and the last layer's twiddles are compile-time constants.  Per transform and
// wave this moves 8 16-byte LDS accesses per lane for the transpose and 4.75 for twiddles,
// where the one-transform form (4 points per lane) moves 16 and 10 and 16 register swaps.
// Every butterfly and twiddle product is the one of fft1024.hpp on the same values, so the
// words are the same.
//
// The cross-wave step: wave r writes its outputs Y_r[k] (k < 256) into its own LDS region;
// after a barrier wave w reads the four waves' values at its 64 k (k's top two bits = w),
// multiplies by T_r[k] and runs the radix-4 over r, so that slot q of wave w holds frequency
// k + 256 q.  Reading each value once (4 accesses per lane and transform instead of 16,
// when every wave read all four inputs for its own quarter of the outputs) also computes
// each radix-4 once (16 additions instead of 32 FMAs per lane).
//
// The exact form's products are rounded to the same integers whatever the order of the FP64
// operations, so its transforms (suffix _pw) fuse the twiddles into the butterflies: a
// radix-4 step whose inputs carry w^0 .. w^3 takes 24 FMAs where three twiddle products and the
// butterfly take 28 operations, and with the twiddles of all steps written as powers (the twist and
// the previous step's factors together) a lane reads 10 per transform instead of 19.  10% fewer
// FP64 operations and 7% fewer LDS accesses per step: exact PBS of 128 inputs 6.63 -> 6.45 ms; at full
// load the clock gives part of it back (1024 inputs 23.3 -> 22.7 ms a round with the HomTrace keys).
// The one-product form's words depend on every rounding, so it keeps the form above.
#pragma once
#include "fft1024.hpp"

namespace tfhe {

constexpr int ROWS_STRIDE = 16 * 17;            // one transform's 16 x 16 transpose, rows padded by one
constexpr int ROWS_CPLX = 4 * ROWS_STRIDE;      // LDS region of one wave

// twiddles in LDS: p1t [4 k0][64 b] as FFT1024Tables, p2 [4 e][16], p3 [4 p][4] (their
// entries depend on the lane mod 16 and mod 4 only)
struct RowTables {
    const cplx* p1t;
    const cplx* p2;
    const cplx* p3;
};
constexpr int ROW_TABLES_CPLX = 256 + 64 + 16;
constexpr int PW_TABLES_CPLX = 160;  // pw as FFT1024Tables

__device__ __forceinline__ RowTables stage_row_tables(const FFT1024Tables& Tg, cplx* tl) {
    for (int k = threadIdx.x; k < 256; k += blockDim.x) tl[k] = Tg.p1t[k];
    for (int k = threadIdx.x; k < 64; k += blockDim.x) tl[256 + k] = Tg.p2[(k >> 4) * 64 + (k & 15)];
    for (int k = threadIdx.x; k < 16; k += blockDim.x) tl[320 + k] = Tg.p3[(k >> 2) * 64 + (k & 3)];
    __syncthreads();
    return {tl, tl + 256, tl + 320};
}

// W16^(h p), h, p in 1..3, the doubles of the p3 table
__device__ __forceinline__ cplx w16_const(int n) {
    constexpr double K[10][2] = {{1.0, 0.0},
                                 {0x1.d906bcf328d46p-1, -0x1.87de2a6aea963p-2},
                                 {0x1.6a09e667f3bcdp-1, -0x1.6a09e667f3bccp-1},
                                 {0x1.87de2a6aea964p-2, -0x1.d906bcf328d46p-1},
                                 {0x1.1a62633145c07p-54, -0x1.0000000000000p+0},
                                 {-0x1.87de2a6aea962p-2, -0x1.d906bcf328d46p-1},
                                 {-0x1.6a09e667f3bccp-1, -0x1.6a09e667f3bcdp-1},
                                 {-0x1.d906bcf328d46p-1, -0x1.87de2a6aea965p-2},
                                 {-0x1.0000000000000p+0, -0x1.1a62633145c07p-53},
                                 {-0x1.d906bcf328d47p-1, 0x1.87de2a6aea961p-2}};
    return {K[n][0], K[n][1]};
}

// position of (lane group index L = 4 k0 + e, p) in a 64-entry block of wave outputs: the
// frequency lane 4 L + p with p swizzled, so that both the writes (fixed p, stride 4) and
// the reads (lane order) touch all banks
__device__ __forceinline__ int row_pos(int L, int p) { return 4 * L + (p ^ ((L >> 1) & 3)); }
__device__ __forceinline__ int row_pos_lane(int lane) { return lane ^ ((lane >> 3) & 3); }

// Forward: x[a][c] at lane 16 R + d = point 64 a + 16 c + d of transform R (untwisted);
// the outputs k = k0 + 4 e + 16 p + 64 s are left in the wave's region at
// [R][s][row_pos(4 k0 + e, p)].  SYNC: a workgroup barrier before the region is first
// written (other waves may still be reading it).
template <bool SYNC>
__device__ __forceinline__ void fft256_fwd_rows(cplx (&x)[4][4], cplx* region, const RowTables& T, int lane) {
    const int R = lane >> 4, d = lane & 15;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        cplx y[4] = {x[0][c], cmul(x[1][c], twist4_const(1)), cmul(x[2][c], twist4_const(2)),
                     cmul(x[3][c], twist4_const(3))};
        dft4<false>(y);
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k][c] = cmul(y[k], T.p1t[k * 64 + 16 * c + d]);
    }
    cplx p2[3];
#pragma unroll
    for (int e = 1; e < 4; ++e) p2[e - 1] = T.p2[e * 16 + d];
    if constexpr (SYNC) lds_barrier();
    cplx* wr = region + R * ROWS_STRIDE + d;
#pragma unroll
    for (int k0 = 0; k0 < 4; ++k0) {
        dft4<false>(x[k0]);
        wr[(4 * k0) * 17] = x[k0][0];
#pragma unroll
        for (int e = 1; e < 4; ++e) wr[(4 * k0 + e) * 17] = cmul(x[k0][e], p2[e - 1]);
    }
    wave_sync();
    const int L = d;  // now 4 k0 + e
    const cplx* rd = region + R * ROWS_STRIDE + L * 17;
    cplx z[4][4];  // [p][h]
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        cplx y[4] = {rd[h], rd[4 + h], rd[8 + h], rd[12 + h]};
        dft4<false>(y);
        z[0][h] = y[0];
#pragma unroll
        for (int p = 1; p < 4; ++p) z[p][h] = h ? cmul(y[p], w16_const(h * p)) : y[p];
    }
    wave_sync();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        dft4<false>(z[p]);
        cplx* o = region + R * 256 + row_pos(L, p);
#pragma unroll
        for (int s = 0; s < 4; ++s) o[s * 64] = z[p][s];
    }
}

// fft256_fwd_rows with the twiddles fused: point b = 64 a + 16 c + d carries v0^b, v0 = w^4, and
// k = k0 + 4 e + 16 p + 64 s.  Over a: powers of v0^64 = exp(i pi / 8).  Over c: of (v0 W256^k0)^16 =
// exp(i pi (1 - 4 k0) / 32).  What is left for d is v^d, v = v0 W256^(k0 + 4 e), one v per lane after
// the transpose (d = 4 g + h): over g powers of v^4, over h powers of v W16^p.  T: pw in LDS.
template <bool SYNC>
__device__ __forceinline__ void fft256_fwd_rows_pw(cplx (&x)[4][4], cplx* region, const cplx* T, int lane) {
    const int R = lane >> 4, d = lane & 15;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        cplx y[4] = {x[0][c], x[1][c], x[2][c], x[3][c]};
        dft4_pw<false>(y, pw_const(4), pw_const(8));
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k][c] = y[k];
    }
    if constexpr (SYNC) lds_barrier();
    cplx* wr = region + R * ROWS_STRIDE + d;
#pragma unroll
    for (int k0 = 0; k0 < 4; ++k0) {
        dft4_pw<false>(x[k0], pw_const(1 - 4 * k0), pw_const(2 - 8 * k0));
#pragma unroll
        for (int e = 0; e < 4; ++e) wr[(4 * k0 + e) * 17] = x[k0][e];
    }
    wave_sync();
    const int L = d;  // now 4 k0 + e
    const cplx* rd = region + R * ROWS_STRIDE + L * 17;
    const cplx t4 = T[L], t8 = T[16 + L];
    cplx z[4][4];  // [p][h]
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        cplx y[4] = {rd[h], rd[4 + h], rd[8 + h], rd[12 + h]};
        dft4_pw<false>(y, t4, t8);
#pragma unroll
        for (int p = 0; p < 4; ++p) z[p][h] = y[p];
    }
    wave_sync();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        dft4_pw<false>(z[p], T[(2 + 2 * p) * 16 + L], T[(3 + 2 * p) * 16 + L]);
        cplx* o = region + R * 256 + row_pos(L, p);
#pragma unroll
        for (int s = 0; s < 4; ++s) o[s * 64] = z[p][s];
    }
}

// Inverse of the same: the region holds [R][s][row_pos(4 k0 + e, p)]; x[a][c] at lane
// 16 R + d returns 256 x the folded point 64 a + 16 c + d of transform R.
__device__ __forceinline__ void fft256_inv_rows(cplx (&x)[4][4], cplx* region, const RowTables& T, int lane) {
    const int R = lane >> 4, d = lane & 15, L = d;
    cplx z[4][4];  // [h][p]
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const cplx* o = region + R * 256 + row_pos(L, p);
        cplx y[4] = {o[0], o[64], o[128], o[192]};
        dft4<true>(y);
#pragma unroll
        for (int h = 0; h < 4; ++h) z[h][p] = y[h];
    }
    wave_sync();
    cplx* wr = region + R * ROWS_STRIDE + L * 17;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        if (h) dft4_pw<true>(z[h], pw_const(4 * h), pw_const(8 * h));  // powers of conj W16^h
        else dft4<true>(z[h]);
#pragma unroll
        for (int g = 0; g < 4; ++g) wr[4 * g + h] = z[h][g];
    }
    wave_sync();
    const cplx* rd = region + R * ROWS_STRIDE + d;
    const cplx w1 = cconj(T.p2[16 + d]), w2 = cconj(T.p2[32 + d]);
#pragma unroll
    for (int k0 = 0; k0 < 4; ++k0) {
        cplx y[4] = {rd[(4 * k0) * 17], rd[(4 * k0 + 1) * 17], rd[(4 * k0 + 2) * 17], rd[(4 * k0 + 3) * 17]};
        dft4_pw<true>(y, w1, w2);
#pragma unroll
        for (int c = 0; c < 4; ++c) x[k0][c] = cmulc(y[c], T.p1t[k0 * 64 + 16 * c + d]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        cplx y[4] = {x[0][c], x[1][c], x[2][c], x[3][c]};
        dft4<true>(y);
        x[0][c] = y[0];
#pragma unroll
        for (int a = 1; a < 4; ++a) x[a][c] = cmulc(y[a], twist4_const(a));
    }
}

// NT inverse 256-point transforms with 4 points per lane (the layout of fft256_inv) side by
// side: the twiddle reads are shared and their LDS round trips overlap.  Slot s of lane
// 16 k0 + 4 e + p in, point 64 a + lane out; region: NT x F256_LDS_CPLX of transposes.
// PW: twiddles fused (the exact form).
template <int NT, bool PW>
__device__ __forceinline__ void fft256_inv_multi(cplx (&x)[NT][4], cplx* region, const RowTables& T, int lane) {
    const int k0 = lane >> 4, e = (lane >> 2) & 3, low = lane & 3, d = lane & 15;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        dft4<true>(x[t]);
#pragma unroll
        for (int hh = 0; hh < 4; ++hh) region[t * F256_LDS_CPLX + f256_a3(k0, e, low, hh)] = x[t][hh];
    }
    wave_sync();
    cplx tw[3];
#pragma unroll
    for (int p = 1; p < 4; ++p) tw[p - 1] = T.p3[p * 4 + low];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < 4; ++p) x[t][p] = region[t * F256_LDS_CPLX + f256_a3(k0, e, p, low)];
    wave_sync();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if constexpr (PW) {
            dft4_pw<true>(x[t], cconj(tw[0]), cconj(tw[1]));
        } else {
#pragma unroll
            for (int p = 1; p < 4; ++p) x[t][p] = cmulc(x[t][p], tw[p - 1]);
            dft4<true>(x[t]);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) region[t * F256_LDS_CPLX + f256_a2(k0, e, 4 * g + low)] = x[t][g];
    }
    wave_sync();
#pragma unroll
    for (int ee = 1; ee < 4; ++ee) tw[ee - 1] = T.p2[ee * 16 + d];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int ee = 0; ee < 4; ++ee) x[t][ee] = region[t * F256_LDS_CPLX + f256_a2(k0, ee, d)];
    wave_sync();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if constexpr (PW) {
            dft4_pw<true>(x[t], cconj(tw[0]), cconj(tw[1]));
        } else {
#pragma unroll
            for (int ee = 1; ee < 4; ++ee) x[t][ee] = cmulc(x[t][ee], tw[ee - 1]);
            dft4<true>(x[t]);
        }
        row_transpose4(x[t]);
    }
    cplx p1[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) p1[k] = T.p1t[k * 64 + lane];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[t][k] = cmulc(x[t][k], p1[k]);
        dft4<true>(x[t]);
#pragma unroll
        for (int a = 1; a < 4; ++a) x[t][a] = cmulc(x[t][a], twist4_const(a));
    }
}

// cross-wave twiddles T_r[k], r = 1..3, of this wave's 64 k (T_0 = 1)
__device__ __forceinline__ void load_cross(const FFT1024Tables& Tg, int w, int lane, cplx (&tr)[3]) {
#pragma unroll
    for (int r = 1; r < 4; ++r) tr[r - 1] = Tg.tr[(r * 4 + w) * 64 + lane];
}

// transform R of the four waves' regions (group: the first wave's region) at this lane's k:
// slot q = frequency k + 256 q; PW: T_r = T_1^r fused
template <bool PW>
__device__ __forceinline__ void cross_fwd(const cplx* group, int R, int w, int lane, const cplx (&tr)[3], cplx (&x)[4]) {
    const cplx* p = group + R * 256 + w * 64 + row_pos_lane(lane);
    if constexpr (PW) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = p[r * ROWS_CPLX];
        dft4_pw<false>(x, tr[0], tr[1]);
    } else {
        x[0] = p[0];
#pragma unroll
        for (int r = 1; r < 4; ++r) x[r] = cmul(p[r * ROWS_CPLX], tr[r - 1]);
        dft4<false>(x);
    }
}

// the inverse radix-4 over q and the conjugate cross twiddles; x[r] belongs to wave r
__device__ __forceinline__ void cross_inv(cplx (&x)[4], const cplx (&tr)[3]) {
    dft4<true>(x);
#pragma unroll
    for (int r = 1; r < 4; ++r) x[r] = cmulc(x[r], tr[r - 1]);
}

// digits of four rows packed (real part low half, imaginary part high half, sign bit of
// each digit flipped into two's complement position) -> two signed values as doubles
template <int LOGB>
__device__ __forceinline__ cplx unpack_digits(uint32_t v) {
    const int32_t re = (int32_t)(v << (32 - LOGB)) >> (32 - LOGB);
    const int32_t im = (int32_t)(v << (16 - LOGB)) >> (32 - LOGB);
    return {(double)re, (double)im};
}

// 4 x 4 transpose of (slot, 16-lane row) of plain words, as row_transpose4
__device__ __forceinline__ void row_transpose4_u32(uint32_t (&d)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto e = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    d[0] = c[0];
    d[1] = c[1];
    d[2] = e[0];
    d[3] = e[1];
}

// The four digit rows of the 8 coefficients a lane owns (point 64 a + lane: acc[a] real,
// acc[a + 4] imaginary), as inputs of fft256_fwd_rows: signed digits in [-B/2, B/2) by the
// offset method, row j = bits IGN + j LOGB.
template <int LOGB>
__device__ __forceinline__ void digit_rows(const uint64_t (&acc)[8], cplx (&x)[4][4]) {
    constexpr int L = 4, IGN = 64 - L * LOGB;
    constexpr uint32_t M = (1u << LOGB) - 1;
    uint64_t off = 1ull << (IGN - 1), flip = 0;
#pragma unroll
    for (int j = 0; j < L; ++j) flip |= (1ull << (LOGB - 1)) << (IGN + j * LOGB);
    off += flip;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const uint64_t re = (acc[a] + off) ^ flip, im = (acc[a + 4] + off) ^ flip;
        uint32_t q[4];
#pragma unroll
        for (int j = 0; j < L; ++j) {
            const uint32_t dr = (uint32_t)(re >> (IGN + j * LOGB)) & M, di = (uint32_t)(im >> (IGN + j * LOGB)) & M;
            q[j] = dr | (di << 16);
        }
        row_transpose4_u32(q);
#pragma unroll
        for (int c = 0; c < 4; ++c) x[a][c] = unpack_digits<LOGB>(q[c]);
    }
}

}  // namespace tfhe
