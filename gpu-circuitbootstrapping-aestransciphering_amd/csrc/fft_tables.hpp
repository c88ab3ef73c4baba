// fft_tables.hpp -- values of the N = 2048 transform's twiddle tables (host code, standard C++).
#pragma once
#include <cmath>
#include <vector>

namespace tfhe {

struct TableValue {
    double re, im;
};
// p1t, p2, p3 [4][64], tr [4][4][64], rot [2N], pw [10][16] of fft1024.hpp, in device order
constexpr int FFT1024_TABLE_CPLX = 1792 + 4096 + 160;

// rounded: sine and cosine rounded once, for the exact PBS, whose products are all rounded to
// integers: their distance from the integers is a quarter smaller (2^10 x 4 gadget: rms 0.028 against
// 0.037).  Otherwise those of the angle in double, off by up to six units in the last place: the
// one-product PBS's words depend on every rounding, and these values are part of them.
inline std::vector<TableValue> fft1024_tables(bool rounded) {
    std::vector<TableValue> h(FFT1024_TABLE_CPLX);
    const double PI = 3.14159265358979323846264338327950288;
    const int N = 2048;
    std::vector<TableValue> oct;  // exp(i pi j / 2048), j <= 512
    if (rounded)
        for (int j = 0; j <= 512; ++j) {
            const long double a = 3.14159265358979323846264338327950288L * j / N;
            oct.push_back({(double)std::cos(a), (double)std::sin(a)});
        }
    // exp(i ang), ang = pi j / 2048 up to turns
    auto put = [&](int idx, double ang, int j) {
        if (!rounded) {
            h[idx] = {std::cos(ang), std::sin(ang)};
            return;
        }
        const int r = j & 1023;
        const TableValue v = r <= 512 ? oct[r] : TableValue{oct[1024 - r].im, oct[1024 - r].re};
        switch ((j >> 10) & 3) {
            case 0: h[idx] = v; break;
            case 1: h[idx] = {-v.im, v.re}; break;
            case 2: h[idx] = {-v.re, -v.im}; break;
            default: h[idx] = {v.im, -v.re};
        }
    };
    for (int k0 = 0; k0 < 4; ++k0)
        for (int b = 0; b < 64; ++b)  // (w^4)^b * W256^(b k0)
            put(k0 * 64 + b, PI * 4.0 * b / N - 2.0 * PI * (double)((b * k0) % 256) / 256.0, 4 * b - 16 * b * k0);
    for (int e = 0; e < 4; ++e)
        for (int L = 0; L < 64; ++L)
            put(256 + e * 64 + L, -2.0 * PI * (double)(((L & 15) * e) % 64) / 64.0, -64 * (L & 15) * e);
    for (int p = 0; p < 4; ++p)
        for (int L = 0; L < 64; ++L)
            put(512 + p * 64 + L, -2.0 * PI * (double)(((L & 3) * p) % 16) / 16.0, -256 * (L & 3) * p);
    for (int r = 0; r < 4; ++r)
        for (int s = 0; s < 4; ++s)
            for (int l = 0; l < 64; ++l) {
                const int k = (l >> 4) + 4 * ((l >> 2) & 3) + 16 * (l & 3) + 64 * s;
                put(768 + (r * 4 + s) * 64 + l, PI * r / N - 2.0 * PI * (double)((r * k) % 1024) / 1024.0, r - 4 * r * k);
            }
    for (int j = 0; j < 2 * N; ++j) put(1792 + j, PI * j / N, j);
    for (int L = 0; L < 16; ++L) {
        const int k = (L >> 2) + 4 * (L & 3);
        auto pw = [&](int t, int p, int power) {  // (w^4 W256^(k + 16 p))^power, in units of pi / 512
            const int num = (1 - 4 * (k + 16 * p)) * power;
            put(1792 + 2 * N + t * 16 + L, PI * (double)(num % 1024) / 512.0, 4 * num);
        };
        pw(0, 0, 4);
        pw(1, 0, 8);
        for (int p = 0; p < 4; ++p) {
            pw(2 + 2 * p, p, 1);
            pw(3 + 2 * p, p, 2);
        }
    }
    return h;
}

}  // namespace tfhe
