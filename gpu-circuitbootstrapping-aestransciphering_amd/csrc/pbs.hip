// pbs.hip -- the multi-value programmable bootstrap (the circuit bootstrap's blind
// rotation), N = 2048 on the 64-bit torus: one workgroup per ciphertext, accumulator in
// registers in the FFT1024 coefficient ownership.  Input LWE_s (torus-32) of b * 2^31.
// Steps (reference ManyLUT path, cirbts-batch.cu:3293-4006, restated for the torus-64 CGGI
// accumulator): b += 2^30; a~_i = special_ms(a_i, bw = 1); test vector with b~ folded in;
// n CMux steps acc += (X^m - 1)(dec(acc) (*) BSK_i), m = -a~_i mod 2N (or n/2 steps over
// key-bit pairs, MB = 2); extract coefficients 0 and 1 and add mu_j = 2^(47 + 8j).
// Output [batch][2][N+1] u64: LWE_K2 of b * 2^(48 + 8j).
#include "cbs_device.hpp"
#include "fft_rows.hpp"
#include "kernels.hpp"

namespace tfhe {

// round(v * 2N / (2^32 2^bw)) * 2^bw mod 2N with N = 2048, bw = 1
__device__ __forceinline__ uint32_t special_ms_2048(uint32_t v) {
    return (uint32_t)((((uint64_t)v + (1ull << 20)) >> 21) << 1) & 4095u;
}
// the same for any bw in [0, 11] (the reference's gpu_SpecilMS, cirbts-utils.cu:52-61)
__device__ __forceinline__ uint32_t special_ms_2048_bw(uint32_t v, uint32_t bw) {
    return (uint32_t)((((uint64_t)v + (1ull << (19 + bw))) >> (20 + bw)) << bw) & 4095u;
}

// c ? a : b by value (a select of the operands' addresses would keep them in memory)
__device__ __forceinline__ cplx csel(int c, cplx a, cplx b) { return {c ? a.re : b.re, c ? a.im : b.im}; }

// coefficient of slot h (h < 4: point 64 h + lane, real; else + N/2, imaginary) of (wave, lane)
__device__ __forceinline__ uint32_t slot_coeff(int w, int lane, int h) {
    return (uint32_t)own_coeff(w, lane, h & 3) + (h >= 4 ? CB_M : 0);
}

// acc + a b, or a b alone for the first product of a sum
__device__ __forceinline__ void cmac_first(bool first, cplx& acc, cplx a, cplx b) {
    if (first) acc = {fma(-a.im, b.im, a.re * b.re), fma(a.im, b.re, a.re * b.im)};
    else cmac(acc, a, b);
}

// What one blind-rotation step multiplies by.
//   LIMBS = 2: BSK2 Fourier rows hold the two signed 32-bit limbs of each torus-64
//     coefficient and every product is rounded exactly.
//   LIMBS = 1: one Fourier row of the coefficients scaled to the torus
//     (k_to_fourier2048_t64); the product is rounded once, to about 2^-36 of the torus per step.
// The monic factor is applied pointwise before the inverse transform: frequency k is the
// polynomial at w^(1 - 4k), so (X^m - 1) multiplies it by w^(m (1 - 4k)) - 1 (one rounding
// of (X^m - 1) t gives the integers of rotating the rounded t).
//   MB = 2 (one limb only): two key bits per step.  With m1, m2 the rotations of the pair,
//     acc += sum_p (X^(e_p) - 1) (dec(acc) (*) RGSW(ind_p)) over the patterns (1,0), (0,1),
//     (1,1) with e_p = m1, m2, m1 + m2: exactly one indicator is 1 (or none), so this equals
//     the two single-bit steps.  One decomposition and two inverse transforms serve both
//     bits; the factor of pattern p is applied to the digit transforms before they meet that
//     pattern's key row.
// The factor of frequency k + 512 is that of k times w^(-2048 m): the same table entry for an
// even rotation m.  The circuit bootstrap's rotations are even (modulus switch with bw = 1), so
// a lane looks up half its factors (a lookup is a gather of one cache line per lane); with a
// caller's bitwidth (ANYM) every factor has its own.
// Key loads come in batches of 8 values per lane (8 KB per wave): MB = 2: one pattern of one
// row for both outputs; LIMBS = 2: one output of one row; else one row for both outputs.
template <int LIMBS, int MB, bool ANYM>
struct PbsStep {
    static_assert(MB == 1 || LIMBS == 1, "two key bits per step only in the one-product form");
    static constexpr int NQ = ANYM ? 4 : 2, FP = MB == 2 ? 3 : 1;
    static constexpr int BPR = MB == 2 ? 3 : LIMBS;                 // batches per digit row
    static constexpr int BATCHES = PBS_L * BPR;                     // per accumulator polynomial
    static constexpr size_t KEY = (size_t)(MB == 2 ? 3 : 1) * PBS_ROWS * 2 * LIMBS * CB_M;  // per step

    // batch t of polynomial u's rows (row r = 2 j + u), outputs first, second (the own and the
    // other group's in the split form).  key is uniform over the wave, at the lane's frequency
    // offset: scalar base addresses, one vector offset for all loads
    static __device__ __forceinline__ void load(cplx (&kv)[2][4], const cplx* key, uint32_t at, int u, int t,
                                                int first, int second) {
        at = fresh_offset(at);
        const int j = t / BPR, b = t % BPR, r = 2 * j + u;
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int out = o ? second : first;
            const cplx* k;
            if constexpr (MB == 2) {
                const int pt = b == 0 ? 0 : b == 1 ? 2 : 1;  // factors in the order (1,0), (1,1), (0,1)
                k = key + ((size_t)(pt * PBS_ROWS + r) * 2 + out) * CB_M;
            } else if constexpr (LIMBS == 2) {  // batch b: output first or second, limb o
                k = key + ((size_t)(r * 2 + (b ? second : first)) * 2 + o) * CB_M;
            } else {
                k = key + ((size_t)r * 2 + out) * CB_M;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) kv[o][q] = key_at(k + q * 256, at);
        }
    }
    // batch t's products; x: the digit transform of its row; fp: pattern factors (MB = 2)
    static __device__ __forceinline__ void mac(cplx (&acc)[2][LIMBS][4], const cplx (&x)[4],
                                               const cplx (&fp)[FP][NQ], const cplx (&kv)[2][4], int t, bool fresh) {
        const bool first = fresh && t < LIMBS;
        const int b = t % BPR;
        if constexpr (MB == 2) {
            cplx y[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) y[q] = cmul(x[q], fp[b][q % NQ]);
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int q = 0; q < 4; ++q) cmac_first(first, acc[o][0][q], y[q], kv[o][q]);
        } else {
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (LIMBS == 2) cmac_first(first, acc[b][o][q], x[q], kv[o][q]);
                    else cmac_first(first, acc[o][0][q], x[q], kv[o][q]);
                }
        }
    }
    // factors of this lane's frequencies (exponents ek) for the step's rotations
    static __device__ __forceinline__ void factors(cplx (&fp)[FP][NQ], const cplx* rot, uint32_t m1, uint32_t m2,
                                                   const uint32_t (&ek)[4]) {
        constexpr uint32_t Q2 = 2 * CB_N;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const cplx z1 = rot[(m1 * ek[q]) & (Q2 - 1)];
            fp[0][q] = {z1.re - 1.0, z1.im};
            if constexpr (MB == 2) {
                const cplx z2 = rot[(m2 * ek[q]) & (Q2 - 1)];
                const cplx z12 = cmul(z1, z2);
                fp[1][q] = {z12.re - 1.0, z12.im};
                fp[2][q] = {z2.re - 1.0, z2.im};
            }
        }
    }
};

// The rows of one accumulator polynomial: transforms are in the group's regions, key batches
// 0 and 1 in flight (ka, kb).  A batch is loaded after the MACs of the batch two before it, so
// two are in flight or in use at a time (64 registers); the scheduling fences keep it so.
template <class S, int LIMBS>
__device__ __forceinline__ void pbs_mac_rows(cplx (&acc)[2][LIMBS][4], const cplx (&fp)[S::FP][S::NQ],
                                             cplx (&ka)[2][4], cplx (&kb)[2][4], const cplx* key, uint32_t at, int u,
                                             bool fresh, int first, int second, const cplx* group, int w, int lane,
                                             const cplx (&tr)[3]) {
    cplx x[4];
#pragma unroll
    for (int t = 0; t < S::BATCHES; ++t) {
        if (t % S::BPR == 0) cross_fwd<LIMBS == 2>(group, t / S::BPR, w, lane, tr, x);
        if (t & 1) S::mac(acc, x, fp, kb, t, fresh);
        else S::mac(acc, x, fp, ka, t, fresh);
        __builtin_amdgcn_sched_barrier(0);
        if (t + 2 < S::BATCHES) {
            if (t & 1) S::load(kb, key, at, u, t + 2, first, second);
            else S::load(ka, key, at, u, t + 2, first, second);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// rotations of the input and the accumulator's start
template <bool LUT>
__device__ __forceinline__ uint32_t pbs_rotations(const uint32_t* ct, int n, uint16_t* at, const PbsLut& io) {
    constexpr uint32_t Q2 = 2 * CB_N;
    uint32_t bt;
    if constexpr (LUT) {
        // rotation by X^{+a~_i s_i} (the step multiplies by X^{-at[i]}), so that acc ends
        // as LUT X^{-phase~}
        for (int k = threadIdx.x; k < n; k += blockDim.x)
            at[k] = (uint16_t)((Q2 - special_ms_2048_bw(ct[k], io.bw)) & (Q2 - 1));
        bt = special_ms_2048_bw(ct[n] + io.b_add, io.bw);
    } else {
        for (int k = threadIdx.x; k < n; k += blockDim.x) at[k] = (uint16_t)special_ms_2048(ct[k]);
        bt = special_ms_2048(ct[n] + (1u << 30));
    }
    return bt;
}
constexpr uint64_t PBS_MU0 = 1ull << 47, PBS_MU1 = 1ull << 55;
// body polynomial's start at coefficient c: LUT X^-bt, or the two-level test vector
template <bool LUT>
__device__ __forceinline__ uint64_t pbs_start(uint32_t c, uint32_t bt, const PbsLut& io) {
    constexpr uint32_t N = CB_N, Q2 = 2 * CB_N;
    if constexpr (LUT) {  // coefficient c is LUT[m], m = c + bt mod 2N, negated for m >= N
        const uint32_t m = (c + bt) & (Q2 - 1);
        const uint64_t v = io.lut[m & (N - 1)];
        return m >= N ? 0 - v : v;
    } else {
        const uint32_t arg = (bt + Q2 - (c & ~1u)) & (Q2 - 1);
        const uint64_t v = 0 - ((c & 1) ? PBS_MU1 : PBS_MU0);
        return arg >= N ? 0 - v : v;
    }
}

// exact form, after fft256_inv_rows: lane group R = 2 o + lb holds limb lb of output o: round,
// move the limb into place, transpose back to the accumulator's ownership and add
__device__ __forceinline__ void add_limb_rows(uint64_t (&acc)[2][8], const cplx (&x)[4][4], int lane, double magic) {
    const int up = (lane & 16) ? 32 : 0;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint64_t v = (uint64_t)round_i64(part ? x[a][c].im : x[a][c].re, 1.0 / CB_M, magic) << up;
                lo[c] = (uint32_t)v;
                hi[c] = (uint32_t)(v >> 32);
            }
            row_transpose4_u32(lo);
            row_transpose4_u32(hi);
#pragma unroll
            for (int o = 0; o < 2; ++o)
                acc[o][a + 4 * part] += (((uint64_t)hi[2 * o] << 32) | lo[2 * o]) + ((uint64_t)hi[2 * o + 1] << 32);
        }
}

// the whole RLWE (mask, body), Gpow_j / 2 added to body coefficient j < 2
__device__ __forceinline__ void pbs_store_rlwe(const uint64_t (&acc)[2][8], int w, int lane, uint64_t* r,
                                               const PbsLut& io) {
    const uint64_t o0 = io.offsets ? PBS_MU0 : 0, o1 = io.offsets ? PBS_MU1 : 0;
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const uint32_t c = slot_coeff(w, lane, h);
        r[c] = acc[0][h];
        r[CB_N + c] = acc[1][h] + (c == 0 ? o0 : c == 1 ? o1 : 0);
    }
}

// sample extraction of coefficients 0 and 1
__device__ __forceinline__ void pbs_extract(const uint64_t (&acc)[2][8], int w, int lane, uint64_t* o0) {
    constexpr uint32_t N = CB_N;
    uint64_t* o1 = o0 + (N + 1);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const uint32_t c = slot_coeff(w, lane, h);
        const uint64_t v = acc[0][h];
        o0[(0u - c) & (N - 1)] = (c == 0) ? v : 0 - v;
        o1[(1u - c) & (N - 1)] = (c <= 1) ? v : 0 - v;
    }
    if (lane == 0 && w == 0) o0[N] = acc[1][0] + PBS_MU0;
    if (lane == 0 && w == 1) o1[N] = acc[1][0] + PBS_MU1;
}

// evaluation exponents 1 - 4k (mod 2N) of this lane's frequencies k = kl + 64 w + 256 q
__device__ __forceinline__ void pbs_exponents(int w, int lane, uint32_t (&ek)[4]) {
    const uint32_t kl = (uint32_t)((lane >> 4) + 4 * ((lane >> 2) & 3) + 16 * (lane & 3) + 64 * w);
#pragma unroll
    for (int q = 0; q < 4; ++q) ek[q] = (1u - 4u * (kl + 256u * (uint32_t)q)) & (2 * CB_N - 1);
}

// L2 prefetch of the next step's keys: workgroups are dealt to the 8 XCDs in turn and run the
// steps nearly in lockstep, so the (up to MAXWG) resident workgroups of one XCD each touch one
// share of the step's 128-byte lines (one word per line), issued after the step's last key
// loads (loads return in order: earlier, the step's own key waits would include it) and
// consumed a step later.
// (THREADS is a constant: blockDim.x would be a load from memory, and a wait for it, per step)
template <size_t KEY_CPLX, uint32_t MAXWG, int PER, uint32_t THREADS>
struct KeyPrefetch {
    static constexpr uint32_t LINES = KEY_CPLX * sizeof(cplx) / 128;
    uint32_t l0, end, pf[PER], sink = 0;
    __device__ __forceinline__ KeyPrefetch() {
        const uint32_t wgs = (gridDim.x + 7) / 8, per_xcd = wgs < MAXWG ? wgs : MAXWG;
        const uint32_t share = (LINES + per_xcd - 1) / per_xcd, part = (blockIdx.x >> 3) % per_xcd;
        end = (part + 1) * share < LINES ? (part + 1) * share : LINES;
        l0 = part * share + threadIdx.x;
#pragma unroll
        for (int k = 0; k < PER; ++k) pf[k] = 0;
    }
    // branch-free: lines past the share are clamped to its last one
    __device__ __forceinline__ void touch(const cplx* key) {
        const char* p = reinterpret_cast<const char*>(key);
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            sink ^= pf[k];  // the previous step's, long landed
            const uint32_t l = l0 + (uint32_t)k * THREADS;
            pf[k] = *reinterpret_cast<const uint32_t*>(p + (size_t)(l < end ? l : end - 1) * 128);
        }
    }
};

// One 4-wave workgroup per ciphertext, two workgroups per CU (77 KB of LDS each): the form of
// the one-bit one-product step, whose key stream (65 KB per wave and step) is short enough
// for two independent workgroups to hide better than two ciphertexts in lockstep do
// (2048 inputs 33.0 ms against 35.2 paired).
template <bool LUT>
__global__ __launch_bounds__(256, 2) void k_pbs2(const uint32_t* __restrict__ lwe, uint32_t batch, int n,
                                                const cplx* __restrict__ bskf, FFT1024Tables Tg,
                                                uint64_t* __restrict__ out, PbsLut io) {
    using S = PbsStep<1, 1, LUT>;
    __shared__ cplx regions[4][ROWS_CPLX];
    __shared__ cplx tl[ROW_TABLES_CPLX];
    __shared__ uint16_t at[1024];
    const RowTables T = stage_row_tables(Tg, tl);
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    cplx tr[3];
    load_cross(Tg, w, lane, tr);
    uint32_t ek[4];
    pbs_exponents(w, lane, ek);
    const double magic = round_magic();
    const uint32_t kat = (uint32_t)(w * 64 + lane) * sizeof(cplx);
    cplx* own = regions[w];
    constexpr uint32_t Q2 = 2 * CB_N;
    KeyPrefetch<S::KEY, 64, 1, 256> next;
    for (uint32_t cidx = blockIdx.x; cidx < batch; cidx += gridDim.x) {
        __syncthreads();
        const uint32_t bt = pbs_rotations<LUT>(lwe + (size_t)cidx * (n + 1), n, at, io);
        __syncthreads();
        uint64_t acc[2][8];
        const int l0 = fresh_lane(lane);
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            acc[0][h] = 0;
            acc[1][h] = pbs_start<LUT>(slot_coeff(w, l0, h), bt, io);
        }
        for (int i = 0; i < n; ++i) {
            const uint32_t m1 = (Q2 - uniform(at[i])) & (Q2 - 1);
            if (m1 == 0) continue;
            const cplx* step = bskf + (size_t)i * S::KEY;
            cplx fp[S::FP][S::NQ];
            cplx macc[2][1][4];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                cplx ka[2][4], kb[2][4];
                {
                    cplx x[4][4];
                    digit_rows<PBS_LOGB>(acc[u], x);
                    // u = 1: the other waves read this wave's region until the barrier; u = 0:
                    // only this wave has used it since the inverse transform's exchange
                    if (u == 0) fft256_fwd_rows<false>(x, own, T, lane);
                    else fft256_fwd_rows<true>(x, own, T, lane);
                }
                S::load(ka, step, kat, u, 0, 0, 1);
                S::load(kb, step, kat, u, 1, 0, 1);
                lds_barrier();
                pbs_mac_rows<S>(macc, fp, ka, kb, step, kat, u, u == 0, 0, 1, &regions[0][0], w, lane, tr);
            }
            next.touch(i + 1 < n ? step + S::KEY : step);
            S::factors(fp, Tg.rot, m1, 0, ek);
#pragma unroll
            for (int o = 0; o < 2; ++o) {
#pragma unroll
                for (int q = 0; q < 4; ++q) macc[o][0][q] = cmul(macc[o][0][q], fp[0][q % S::NQ]);
                cross_inv(macc[o][0], tr);
            }
            lds_barrier();  // every wave has read the digit transforms
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int r = 0; r < 4; ++r) regions[r][o * 256 + w * 64 + lane] = macc[o][0][r];
            lds_barrier();
            cplx y[2][4];
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int s = 0; s < 4; ++s) y[o][s] = own[o * 256 + s * 64 + lane];
            wave_sync();
            fft256_inv_multi<2, false>(y, own, T, lane);
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    acc[o][a] += torus64_from_double(y[o][a].re, magic);
                    acc[o][a + 4] += torus64_from_double(y[o][a].im, magic);
                }
        }
        const int l1 = fresh_lane(lane);
        if constexpr (LUT) pbs_store_rlwe(acc, w, l1, io.rlwe + (size_t)cidx * 2 * CB_N, io);
        else pbs_extract(acc, w, l1, out + (size_t)cidx * 2 * (CB_N + 1));
    }
    if (n < 0) out[threadIdx.x] = next.sink;  // never (n > 0): keeps the prefetch loads
}

// Two ciphertexts per 8-wave workgroup.  Transforms: waves 4c .. 4c + 3 run ciphertext c's.
// Products: wave wv owns the frequencies k + 256 q, k's top two bits = wv & 3, q = hp, hp + 2
// with hp = wv >> 2, of BOTH ciphertexts, so that one key load feeds two products: the key
// stream (196 KB per wave and step in the two-bit form when each ciphertext loads its own) is
// what a step waits on most at this size of launch.
// A wave runs its products and inverse transforms at a higher priority than its forward ones: left
// to the SIMD's order by age, the older of its two waves ran a whole forward transform ahead of the
// younger one's inverse, which then ran alone (17 blocks 283.5 -> 280.4 ms; exact, 8 blocks, 352.9 -> 350.0).
template <int LIMBS, int MB, bool ANYM>
struct PbsPair {
    using S = PbsStep<LIMBS, MB, ANYM>;
    static_assert((LIMBS == 2) != (MB == 2), "the exact or the two-bit step: one limb and one bit run k_pbs2");
    static constexpr int NQ = ANYM ? 2 : 1;
    static constexpr int DEPTH = MB == 2 ? 2 : 4;  // key batches in flight
    cplx macc[2][2][LIMBS][2];       // [ciphertext][output][limb][q]
    cplx fp[2][S::FP][NQ];

    static __device__ __forceinline__ void load(cplx (&kv)[4], const cplx* key, uint32_t at, int u, int t) {
        at = fresh_offset(at);
        const int j = t / S::BPR, b = t % S::BPR, r = 2 * j + u;
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const cplx* k;
            if constexpr (MB == 2) {
                const int pt = b == 0 ? 0 : b == 1 ? 2 : 1;  // factors in the order (1,0), (1,1), (0,1)
                k = key + ((size_t)(pt * PBS_ROWS + r) * 2 + o) * CB_M;
            } else {  // batch b: output b, limb o
                k = key + ((size_t)(r * 2 + b) * 2 + o) * CB_M;
            }
            kv[2 * o] = key_at(k, at);
            kv[2 * o + 1] = key_at(k + 512, at);
        }
    }
    __device__ __forceinline__ void mac(const cplx (&x)[2][2], const cplx (&kv)[4], int u, int t) {
        const int b = t % S::BPR;
        const bool first = u == 0 && t < LIMBS;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if constexpr (MB == 2) {
                    const cplx y = cmul(x[c][q], fp[c][b][q % NQ]);
#pragma unroll
                    for (int o = 0; o < 2; ++o) cmac_first(first, macc[c][o][0][q], y, kv[2 * o + q]);
                } else {
#pragma unroll
                    for (int o = 0; o < 2; ++o) cmac_first(first, macc[c][b][o][q], x[c][q], kv[2 * o + q]);
                }
            }
    }
    __device__ __forceinline__ void factors(const cplx* rot, int c, uint32_t m1, uint32_t m2, const uint32_t (&ek)[2]) {
        constexpr uint32_t Q2 = 2 * CB_N;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const cplx z1 = rot[(m1 * ek[q]) & (Q2 - 1)];
            fp[c][0][q] = {z1.re - 1.0, z1.im};
            if constexpr (MB == 2) {
                const cplx z2 = rot[(m2 * ek[q]) & (Q2 - 1)];
                const cplx z12 = cmul(z1, z2);
                fp[c][1][q] = {z12.re - 1.0, z12.im};
                fp[c][2][q] = {z2.re - 1.0, z2.im};
            }
        }
    }
};

template <int LIMBS, int MB, bool LUT, int LOGB = PBS_LOGB>
__global__ __launch_bounds__(512, 1) void k_pbs2_pair(const uint32_t* __restrict__ lwe, uint32_t batch, int n,
                                                     const cplx* __restrict__ bskf, FFT1024Tables Tg,
                                                     uint64_t* __restrict__ out, PbsLut io) {
    using S = PbsStep<LIMBS, MB, LUT>;
    using P = PbsPair<LIMBS, MB, LUT>;
    __shared__ cplx regions[8][ROWS_CPLX];
    __shared__ cplx tl[ROW_TABLES_CPLX];
    __shared__ uint16_t at[2][1024];
    __shared__ cplx tpw[LIMBS == 2 ? PW_TABLES_CPLX : 1];
    if constexpr (LIMBS == 2)
        for (int k = threadIdx.x; k < PW_TABLES_CPLX; k += blockDim.x) tpw[k] = Tg.pw[k];
    const RowTables T = stage_row_tables(Tg, tl);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cc = wv >> 2, w = wv & 3;  // cc: the transforms' ciphertext, and hp of the products
    // Cross twiddles of the products' frequencies: the radix-4 outputs q and q + 2 are
    // (y0 + e y2) +- W (y1 + e y3), e = 1, W = 1 for q = 0 and e = -1, W = -i for q = 1; e and W
    // folded into the twiddles (multiplying a product's twiddle by -1 or -i moves its exact
    // result, so the words stay those of dft4)
    cplx trf[3];
    {
        cplx tr[3];
        load_cross(Tg, w, lane, tr);
        trf[0] = csel(cc, {tr[0].im, -tr[0].re}, tr[0]);
        trf[1] = csel(cc, {-tr[1].re, -tr[1].im}, tr[1]);
        trf[2] = csel(cc, {-tr[2].im, tr[2].re}, tr[2]);
    }
    uint32_t ek[2];
    {
        uint32_t e4[4];
        pbs_exponents(w, lane, e4);
        ek[0] = cc ? e4[1] : e4[0];
        ek[1] = cc ? e4[3] : e4[2];
    }
    const double magic = round_magic();
    const uint32_t kat = (uint32_t)(wv * 64 + lane) * sizeof(cplx);
    cplx* own = regions[wv];
    cplx* group = regions[4 * cc];
    constexpr uint32_t N = CB_N, Q2 = 2 * CB_N;
    static_assert(LOGB == PBS_LOGB || (LUT && LIMBS == 2), "the 2^10 gadget: exact LUT-mode form only");
    KeyPrefetch<S::KEY, 32, 1, 512> next;
    const uint32_t pairs = (batch + 1) / 2;
    for (uint32_t pidx = blockIdx.x; pidx < pairs; pidx += gridDim.x) {
        // an odd batch's last workgroup runs its ciphertext twice and stores it once
        const uint32_t c0 = 2 * pidx, c1 = c0 + 1 < batch ? c0 + 1 : c0;
        const uint32_t cidx = cc ? c1 : c0;
        __syncthreads();
        const uint32_t b0 = pbs_rotations<LUT>(lwe + (size_t)c0 * (n + 1), n, at[0], io);
        const uint32_t b1 = pbs_rotations<LUT>(lwe + (size_t)c1 * (n + 1), n, at[1], io);
        const uint32_t bt = cc ? b1 : b0;
        __syncthreads();
        uint64_t acc[2][8];
        const int l0 = fresh_lane(lane);
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            acc[0][h] = 0;
            acc[1][h] = pbs_start<LUT>(slot_coeff(w, l0, h), bt, io);
        }
        for (int i = 0; i < n; i += MB) {
            uint32_t m1[2], m2[2] = {0, 0};
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                m1[c] = (Q2 - uniform(at[c ^ cc][i])) & (Q2 - 1);
                if constexpr (MB == 2) m2[c] = (Q2 - uniform(at[c ^ cc][i + 1])) & (Q2 - 1);
            }
            // (a ciphertext alone without a rotation adds zero: its factors are exactly 0)
            if ((m1[0] | m1[1] | m2[0] | m2[1]) == 0) continue;
            const cplx* step = bskf + (size_t)(i / MB) * S::KEY;
            P pr;
            __builtin_amdgcn_s_setprio(0);
            if constexpr (MB == 2 && !LUT) {
#pragma unroll
                for (int c = 0; c < 2; ++c) pr.factors(Tg.rot, c, m1[c], m2[c], ek);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                {
                    cplx x[4][4];
                    digit_rows<LOGB>(acc[u], x);
                    // u = 1: the other waves read this wave's region until the barrier; u = 0:
                    // only this wave has used it since the inverse transform's exchange
                    if constexpr (LIMBS == 2) {
                        if (u == 0) fft256_fwd_rows_pw<false>(x, own, tpw, lane);
                        else fft256_fwd_rows_pw<true>(x, own, tpw, lane);
                    } else {
                        if (u == 0) fft256_fwd_rows<false>(x, own, T, lane);
                        else fft256_fwd_rows<true>(x, own, T, lane);
                    }
                }
                cplx kv[P::DEPTH][4];
#pragma unroll
                for (int t = 0; t < P::DEPTH; ++t) P::load(kv[t], step, kat, u, t);
                if constexpr (MB == 2 && LUT) {
                    // formed for each polynomial: they would hold 48 registers over the transforms
#pragma unroll
                    for (int c = 0; c < 2; ++c) pr.factors(Tg.rot, c, fresh_uniform(m1[c]), fresh_uniform(m2[c]), ek);
                }
                __builtin_amdgcn_s_setprio(2);
                lds_barrier();
                const int rd = w * 64 + row_pos_lane(lane);
                cplx x[2][2];
#pragma unroll
                for (int t = 0; t < S::BATCHES; ++t) {
                    if (t % S::BPR == 0) {
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            const cplx* p = &regions[4 * (c ^ cc)][rd + (t / S::BPR) * 256];
                            if constexpr (LIMBS == 2) {  // T_3 = T_1 T_2
                                const cplx a = cfma(p[0], trf[1], p[2 * ROWS_CPLX]);
                                const cplx b = cfma(p[ROWS_CPLX], trf[1], p[3 * ROWS_CPLX]);
                                x[c][0] = cfma(a, trf[0], b);
                                x[c][1] = twice_less(a, x[c][0]);
                            } else {
                                const cplx a = cadd(p[0], cmul(p[2 * ROWS_CPLX], trf[1]));
                                const cplx b = cadd(cmul(p[ROWS_CPLX], trf[0]), cmul(p[3 * ROWS_CPLX], trf[2]));
                                x[c][0] = cadd(a, b);
                                x[c][1] = csub(a, b);
                            }
                        }
                    }
                    pr.mac(x, kv[t % P::DEPTH], u, t);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + P::DEPTH < S::BATCHES) P::load(kv[t % P::DEPTH], step, kat, u, t + P::DEPTH);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (u == 0) __builtin_amdgcn_s_setprio(0);
            }
            next.touch(i + MB < n ? step + S::KEY : step);
            if constexpr (MB == 1) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    pr.factors(Tg.rot, c, m1[c], 0, ek);
#pragma unroll
                    for (int o = 0; o < 2; ++o)
#pragma unroll
                        for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                            for (int q = 0; q < 2; ++q)
                                pr.macc[c][o][lb][q] = cmul(pr.macc[c][o][lb][q], pr.fp[c][0][q % P::NQ]);
                }
            }
            // each wave gives the other ciphertext's sums to wave wv ^ 4 and gets its own
            // ciphertext's other two q from it
            lds_barrier();  // every wave has read the digit transforms
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                    for (int q = 0; q < 2; ++q) own[((o * LIMBS + lb) * 2 + q) * 64 + lane] = pr.macc[1][o][lb][q];
            lds_barrier();
            // the inverse radix-4 over q with the conjugate cross twiddles (cross_inv); z[r] belongs
            // to wave r.  This wave's sums m are q = hp, hp + 2, the partner's g the other two
            cplx z[2][LIMBS][4];
            const cplx* oth = regions[wv ^ 4];
            const int cx = (int)fresh_uniform((uint32_t)cc);
            const cplx t1 = csel(cx, {-trf[0].im, trf[0].re}, trf[0]), t3 = csel(cx, {trf[2].im, -trf[2].re}, trf[2]);
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int lb = 0; lb < LIMBS; ++lb) {
                    const cplx g0 = oth[((o * LIMBS + lb) * 2) * 64 + lane], g1 = oth[((o * LIMBS + lb) * 2 + 1) * 64 + lane];
                    const cplx m0 = pr.macc[0][o][lb][0], m1s = pr.macc[0][o][lb][1];
                    const cplx sm = cadd(m0, m1s), dm = csub(m0, m1s), sg = cadd(g0, g1), dg = csub(g0, g1);
                    const cplx e = csel(cx, dg, dm), d = mul_mi<true>(csel(cx, dm, dg));
                    z[o][lb][0] = cadd(sm, sg);
                    z[o][lb][1] = cmulc(cadd(e, d), t1);
                    z[o][lb][2] = cmulc(csub(sm, sg), trf[1]);  // -1 of hp = 1 is in the twiddle
                    z[o][lb][3] = cmulc(csub(e, d), t3);
                }
            if constexpr (LIMBS == 1) {
                // the exchange in the regions' second half: the first still holds what the
                // partner reads
#pragma unroll
                for (int o = 0; o < 2; ++o)
#pragma unroll
                    for (int r = 0; r < 4; ++r) group[r * ROWS_CPLX + 512 + o * 256 + w * 64 + lane] = z[o][0][r];
                lds_barrier();
                cplx y[2][4];
#pragma unroll
                for (int o = 0; o < 2; ++o)
#pragma unroll
                    for (int s = 0; s < 4; ++s) y[o][s] = own[512 + o * 256 + s * 64 + lane];
                wave_sync();
                fft256_inv_multi<2, false>(y, own, T, lane);
#pragma unroll
                for (int o = 0; o < 2; ++o)
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        acc[o][a] += torus64_from_double(y[o][a].re, magic);
                        acc[o][a + 4] += torus64_from_double(y[o][a].im, magic);
                    }
            } else {
                lds_barrier();  // the partner has read its sums
                const int pos = w * 64 + row_pos_lane(lane);
#pragma unroll
                for (int o = 0; o < 2; ++o)
#pragma unroll
                    for (int lb = 0; lb < 2; ++lb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) group[r * ROWS_CPLX + (2 * o + lb) * 256 + pos] = z[o][lb][r];
                lds_barrier();
                cplx x[4][4];
                fft256_inv_rows(x, own, T, lane);
                add_limb_rows(acc, x, lane, magic);
            }
        }
        const int l1 = fresh_lane(lane);
        if (cc && c0 + 1 >= batch) continue;  // the repeated ciphertext
        if constexpr (LUT) pbs_store_rlwe(acc, w, l1, io.rlwe + (size_t)cidx * 2 * N, io);
        else pbs_extract(acc, w, l1, out + (size_t)cidx * 2 * (N + 1));
    }
    if (n < 0) out[threadIdx.x] = next.sink;  // never (n > 0): keeps the prefetch loads
}

// One ciphertext per 8-wave workgroup: wave group g (waves 4g .. 4g + 3) owns accumulator
// polynomial g.  Per step each group transforms its polynomial's four digit rows together and
// sums both outputs' products over them; the partial sum of the other group's output goes
// through LDS, and each group inverse-transforms its own output and updates its polynomial.
// A wave runs half the transforms and MACs of the 4-wave form per step, and a CU holds two
// waves per SIMD with one workgroup: the form for launches of at most one workgroup per CU.
// A step is bound by the key stream into the CU (64 bytes per clock: 12.3 k of the two-bit step's
// 25 k clocks, 8.2 k of the exact one's 24 k) and by the transforms, one after the other as long as
// all waves meet before the products.  A group's products need only its own transforms, so the
// groups meet by themselves there (wave_group_barrier): the group whose waves are older on their
// SIMDs streams its keys while the other transforms.  1-block AES-128 CTR fast 37.6 -> 34.0 ms, exact
// 83.9 -> 77.4; 256 inputs fast 4.45 -> 4.29, HomTrace + SchemeSwitch 72.0 -> 66.6.
// Each output's sum is the two groups' partial sums added once, where the 4-wave form runs
// one sum over all eight rows: the same words in the exact form; in the two-bit one-product
// form they differ by FP64 rounding (the phases agree within that form's bound).
template <int LIMBS, int MB, bool LUT, int LOGB = PBS_LOGB>
__global__ __launch_bounds__(512, 1) void k_pbs2_split(const uint32_t* __restrict__ lwe, uint32_t batch, int n,
                                                      const cplx* __restrict__ bskf, FFT1024Tables Tg,
                                                      uint64_t* __restrict__ out, PbsLut io, uint32_t xcds) {
    using S = PbsStep<LIMBS, MB, LUT>;
    // workgroups are dealt to the 8 XCDs in turn; those of the first xcds take the ciphertexts
    if (blockIdx.x % 8 >= xcds) return;
    const uint32_t first = xcds < 8 ? blockIdx.x / 8 * xcds + blockIdx.x % 8 : blockIdx.x;
    const uint32_t stride = xcds < 8 ? gridDim.x / 8 * xcds : gridDim.x;
    __shared__ cplx regions[8][ROWS_CPLX];
    __shared__ cplx tl[ROW_TABLES_CPLX];
    __shared__ uint16_t at[1024];
    __shared__ cplx tpw[LIMBS == 2 ? PW_TABLES_CPLX : 1];
    if constexpr (LIMBS == 2)
        for (int k = threadIdx.x; k < PW_TABLES_CPLX; k += blockDim.x) tpw[k] = Tg.pw[k];
    __shared__ uint32_t arrived[2];  // of each group, for its own barriers
    if (threadIdx.x < 2) arrived[threadIdx.x] = 0;
    const RowTables T = stage_row_tables(Tg, tl);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = wv >> 2, w = wv & 3;
    cplx tr[3];
    load_cross(Tg, w, lane, tr);
    uint32_t ek[4];
    pbs_exponents(w, lane, ek);
    const double magic = round_magic();
    const uint32_t kat = (uint32_t)(w * 64 + lane) * sizeof(cplx);
    cplx* own = regions[wv];
    cplx* group = regions[4 * g];
    constexpr uint32_t N = CB_N, Q2 = 2 * CB_N;
    KeyPrefetch<S::KEY, 16, 2, 512> next;
    uint32_t arrivals = 0;
    if (g) __builtin_amdgcn_s_setprio(1);  // one group ahead of the other (1 block fast 34.0 -> 33.4 ms, exact 77.8 -> 77.1)
    for (uint32_t cidx = first; cidx < batch; cidx += stride) {
        __syncthreads();
        const uint32_t bt = pbs_rotations<LUT>(lwe + (size_t)cidx * (n + 1), n, at, io);
        __syncthreads();
        uint64_t acc[8];  // polynomial g
        const int l0 = fresh_lane(lane);
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            const uint64_t v = pbs_start<LUT>(slot_coeff(w, l0, h), bt, io);
            acc[h] = g ? v : 0;
        }
        for (int i = 0; i < n; i += MB) {
            const uint32_t m1 = (Q2 - uniform(at[i])) & (Q2 - 1);
            uint32_t m2 = 0;
            if constexpr (MB == 2) m2 = (Q2 - uniform(at[i + 1])) & (Q2 - 1);
            if ((m1 | m2) == 0) continue;
            const cplx* step = bskf + (size_t)(i / MB) * S::KEY;
            cplx fp[S::FP][S::NQ];
            if constexpr (MB == 2) S::factors(fp, Tg.rot, m1, m2, ek);
            cplx macc[2][LIMBS][4];  // this group's output, the other group's
            cplx ka[2][4], kb[2][4];
            {
                cplx x[4][4];
                digit_rows<LOGB>(acc, x);
                if constexpr (LIMBS == 2) fft256_fwd_rows_pw<false>(x, own, tpw, lane);
                else fft256_fwd_rows<false>(x, own, T, lane);
            }
            S::load(ka, step, kat, g, 0, g, 1 - g);
            S::load(kb, step, kat, g, 1, g, 1 - g);
            wave_group_barrier(&arrived[g], arrivals += 4);
            pbs_mac_rows<S>(macc, fp, ka, kb, step, kat, g, true, g, 1 - g, group, w, lane, tr);
            next.touch(i + MB < n ? step + S::KEY : step);
            wave_group_barrier(&arrived[g], arrivals += 4);  // the group has read its digit transforms
#pragma unroll
            for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                for (int q = 0; q < 4; ++q) own[(lb * 4 + q) * 64 + lane] = macc[1][lb][q];
            lds_barrier();
            const cplx* oth = regions[4 * (1 - g) + w];
#pragma unroll
            for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                for (int q = 0; q < 4; ++q) macc[0][lb][q] = cadd(macc[0][lb][q], oth[(lb * 4 + q) * 64 + lane]);
            if constexpr (MB == 1) {
                S::factors(fp, Tg.rot, m1, 0, ek);
#pragma unroll
                for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                    for (int q = 0; q < 4; ++q) macc[0][lb][q] = cmul(macc[0][lb][q], fp[0][q % S::NQ]);
            }
            // the exchange of the inverse transform in the regions' second half (the first still
            // holds the partial sums that the other group reads)
#pragma unroll
            for (int lb = 0; lb < LIMBS; ++lb) {
                cross_inv(macc[0][lb], tr);
#pragma unroll
                for (int r = 0; r < 4; ++r) group[r * ROWS_CPLX + 512 + lb * 256 + w * 64 + lane] = macc[0][lb][r];
            }
            lds_barrier();
            cplx y[LIMBS][4];
#pragma unroll
            for (int lb = 0; lb < LIMBS; ++lb)
#pragma unroll
                for (int s = 0; s < 4; ++s) y[lb][s] = own[512 + lb * 256 + s * 64 + lane];
            wave_sync();
            fft256_inv_multi<LIMBS, LIMBS == 2>(y, own, T, lane);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if constexpr (LIMBS == 1) {
                    acc[a] += torus64_from_double(y[0][a].re, magic);
                    acc[a + 4] += torus64_from_double(y[0][a].im, magic);
                } else {
                    acc[a] += (uint64_t)round_i64(y[0][a].re, 1.0 / CB_M, magic) +
                              ((uint64_t)round_i64(y[LIMBS - 1][a].re, 1.0 / CB_M, magic) << 32);
                    acc[a + 4] += (uint64_t)round_i64(y[0][a].im, 1.0 / CB_M, magic) +
                                  ((uint64_t)round_i64(y[LIMBS - 1][a].im, 1.0 / CB_M, magic) << 32);
                }
            }
        }
        const int l1 = fresh_lane(lane);
        if constexpr (LUT) {
            uint64_t* r = io.rlwe + (size_t)cidx * 2 * N;
            const uint64_t o0 = io.offsets ? PBS_MU0 : 0, o1 = io.offsets ? PBS_MU1 : 0;
#pragma unroll
            for (int h = 0; h < 8; ++h) {
                const uint32_t c = slot_coeff(w, l1, h);
                r[g * N + c] = acc[h] + (g && c == 0 ? o0 : g && c == 1 ? o1 : 0);
            }
            continue;
        }
        uint64_t* o0 = out + (size_t)cidx * 2 * (N + 1);
        uint64_t* o1 = o0 + (N + 1);
        if (g == 0) {  // sample extraction of coefficients 0 and 1 from the mask polynomial
#pragma unroll
            for (int h = 0; h < 8; ++h) {
                const uint32_t c = slot_coeff(w, l1, h);
                const uint64_t v = acc[h];
                o0[(0u - c) & (N - 1)] = (c == 0) ? v : 0 - v;
                o1[(1u - c) & (N - 1)] = (c <= 1) ? v : 0 - v;
            }
        } else {  // bodies: coefficient 0 sits in wave 0, coefficient 1 in wave 1 (lane 0, h = 0)
            if (lane == 0 && w == 0) o0[N] = acc[0] + PBS_MU0;
            if (lane == 0 && w == 1) o1[N] = acc[0] + PBS_MU1;
        }
    }
    if (n < 0) out[threadIdx.x] = next.sink;  // never (n > 0): keeps the prefetch loads
}

// ===========================================================================
// Host launchers
// ===========================================================================
int pbs_model_form(uint32_t batch, int limbs, int mb) {
    // Split over 8 waves (one limb, two bits: form 2; two limbs: form 1) up to one workgroup
    // per CU (256 of them), else two ciphertexts per workgroup (form 0): a second round of the split form, 3.3 ms for
    // 256 inputs (exact 5.9), costs more than the paired form's one round of 512, 5.6 (10.8).
    if (mb == 2) return batch <= 256 ? 2 : 0;
    if (limbs == 2) return batch <= 256 ? 1 : 0;
    return 1;
}

template <bool LUT>
static void launch_pbs2_t(const uint32_t* lwe, uint32_t batch, int n, const cplx* bskf, int limbs, int mb,
                          const FFT1024Tables& T, uint64_t* out, hipStream_t st, int form, const PbsLut& io) {
    if (!batch) return;
    const unsigned grid = batch < 2048 ? batch : 2048;  // one workgroup per ciphertext (or pair) at a time
    const unsigned pairs = (batch + 1) / 2, pgrid = pairs < 2048 ? pairs : 2048;
    // The split form of up to 64 ciphertexts runs on as many XCDs as give each 16: the workgroups of
    // an XCD share its L2 and the prefetch of the key stream, which one or two alone would wait for
    // from memory (two-bit, whole call with lookups: 8 inputs 5.16 -> 3.66 ms, 16 4.74 -> 3.55, 32
    // 4.02 -> 3.45, 64 3.47 -> 3.43, 96 the same; exact: 8 9.54 -> 7.58, 32 7.55 -> 7.30, 112 7.77 against 7.9)
    const unsigned xcds = batch > 64 ? 8 : (batch + 15) / 16;
    const unsigned sgrid = xcds < 8 ? (batch + xcds - 1) / xcds * 8 : grid;
    if (form < 0) form = pbs_model_form(batch, limbs, mb);
    if constexpr (LUT) {
        if (limbs == 2 && io.logB == 10) {  // the HomTrace + SchemeSwitch form's 2^10 x 4 gadget
            if (form == 1) k_pbs2_split<2, 1, true, 10><<<sgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io, xcds);
            else k_pbs2_pair<2, 1, true, 10><<<pgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io);
            return;
        }
    }
    if (limbs == 2) {
        if (form == 1) k_pbs2_split<2, 1, LUT><<<sgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io, xcds);
        else k_pbs2_pair<2, 1, LUT><<<pgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io);
    } else if (mb == 1) {
        k_pbs2<LUT><<<grid, 256, 0, st>>>(lwe, batch, n, bskf, T, out, io);
    } else if (form == 2) {
        k_pbs2_split<1, 2, LUT><<<sgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io, xcds);
    } else {
        k_pbs2_pair<1, 2, LUT><<<pgrid, 512, 0, st>>>(lwe, batch, n, bskf, T, out, io);
    }
}

void launch_pbs2(const uint32_t* lwe, uint32_t batch, int n, const cplx* bskf, int limbs, int mb,
                 const FFT1024Tables& T, uint64_t* out, hipStream_t st, int form, const PbsLut& io) {
    if (io.lut)
        launch_pbs2_t<true>(lwe, batch, n, bskf, limbs, mb, T, out, st, form, io);
    else
        launch_pbs2_t<false>(lwe, batch, n, bskf, limbs, mb, T, out, st, form, io);
}

}  // namespace tfhe
