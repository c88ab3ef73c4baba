// cbs_device.hpp -- device helpers shared by the kernels of the circuit-bootstrapping level.
#pragma once
#include "fft1024.hpp"

namespace tfhe {

constexpr int CB_N = 2048, CB_M = 1024;
// PBS gadget: PBS_L = 4 levels of 2^LOGB (LOGB = 9 for every PFKS form, 10 for the
// HomTrace + SchemeSwitch form), the low 64 - 4 LOGB bits dropped with rounding
constexpr int PBS_LOGB = 9, PBS_L = 4, PBS_ROWS = 8;

// signed digits by the offset method on 64 bits: off = 2^(IGN-1) + sum_j (B/2) 2^(IGN + j logB)
template <int LOGB, int L>
__device__ __forceinline__ uint64_t digit_offset64() {
    constexpr int IGN = 64 - L * LOGB;
    uint64_t off = 1ull << (IGN - 1);
#pragma unroll
    for (int j = 0; j < L; ++j) off += (1ull << (LOGB - 1)) << (IGN + j * LOGB);
    return off;
}
template <int LOGB, int L>
__device__ __forceinline__ double digit64(uint64_t tp, int j) {
    constexpr int IGN = 64 - L * LOGB;
    return (double)((int32_t)((tp >> (IGN + j * LOGB)) & ((1u << LOGB) - 1)) - (1 << (LOGB - 1)));
}

// round(y * 2^64) mod 2^64 for a torus value held as a double.  f = y - rint(y)
// in [-1/2, 1/2] is exact; its top 32 bits are rint(f 2^32), taken with the
// 1.5 * 2^52 rounding constant, and the exact residual r = f 2^32 - rint(f 2^32)
// gives the low 32 bits the same way (borrowing one from the top half when
// rint(r 2^32) < 0, i.e. l < MAGIC).
__device__ __forceinline__ uint64_t torus64_from_double(double y, double MAGIC = ROUND_MAGIC) {
    constexpr double TWO32 = 4294967296.0;
    const double f = y - rint(y);
    const double h = fma(f, TWO32, MAGIC);
    const double r = fma(f, TWO32, -(h - MAGIC));
    const double l = fma(r, TWO32, MAGIC);
    const uint32_t hi = (uint32_t)__double_as_longlong(h) - (l < MAGIC ? 1u : 0u);
    return ((uint64_t)hi << 32) | (uint32_t)__double_as_longlong(l);
}

}  // namespace tfhe
