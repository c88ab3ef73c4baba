// capi_common.hpp -- error reporting, device allocation and FFT twiddle tables
// shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/tfhe_amd.h"
#include "device_common.hpp"
#include "fft1024.hpp"
#include "fft512_pair.hpp"
#include "fft_tables.hpp"

namespace tfhe {

int fail(int code, const std::string& msg);
int hipcheck(hipError_t e, const char* what);
int check_launch(const char* what);
int dmalloc(void** p, size_t bytes);

// Twiddle tables of the wavefront FFT (see device_common.hpp for the layout).
struct DeviceTables {
    FFTTables T{};
    cplx* d_buf = nullptr;
    int init(int N) {
        if (N != 1024) return fail(TFHE_E_PARAM, "FFT tables: only N = 1024 is built");
        std::vector<cplx> h(1024 + 2 * N + 1024 + PAIR_TABLE_CPLX + 6 * 64);
        const double PI = 3.14159265358979323846264338327950288;
        for (int k = 0; k < 8; ++k)
            for (int b = 0; b < 64; ++b) {
                // w^b * exp(-2 pi i b k / 512), w = exp(i pi / N)
                const double ang = PI * b / N - 2.0 * PI * (double)((b * k) % 512) / 512.0;
                h[k * 64 + b] = {std::cos(ang), std::sin(ang)};
            }
        for (int e = 0; e < 8; ++e)
            for (int l = 0; l < 64; ++l) {
                const double ang = -2.0 * PI * (double)(((l & 7) * e) % 64) / 64.0;
                h[512 + e * 64 + l] = {std::cos(ang), std::sin(ang)};
            }
        for (int j = 0; j < 2 * N; ++j) {  // w^j, the evaluation points' powers
            const double ang = PI * j / N;
            h[1024 + j] = {std::cos(ang), std::sin(ang)};
        }
        // the two-wave transform: the 256-point step's tables as DeviceTables1024 has them (its
        // twist exp(4 i pi / 2048) is this one's w^2), then w W512^k, k < 256
        cplx* h2 = h.data() + 1024 + 2 * N;
        for (int k = 0; k < 4; ++k)
            for (int l = 0; l < 64; ++l) {
                auto put = [&](int idx, double ang) { h2[idx + k * 64 + l] = {std::cos(ang), std::sin(ang)}; };
                put(0, PI * l / 512.0 - 2.0 * PI * (double)((l * k) % 256) / 256.0);
                put(256, -2.0 * PI * (double)(((l & 15) * k) % 64) / 64.0);
                put(512, -2.0 * PI * (double)(((l & 3) * k) % 16) / 16.0);
                put(768, PI / N - 2.0 * PI * (double)(64 * k + l) / 512.0);
            }
        // the two-transforms-per-wave form (fft512_pair.hpp): square roots down the tree below
        // node n = (b1 b2 b3 b4), whose root angle is th
        cplx* h3 = h2 + 1024;
        for (int n = 0; n < 16; ++n) {
            const double th = PI / 32 + PI * (((n >> 3) & 1) / 8.0 + ((n >> 2) & 1) / 4.0 + ((n >> 1) & 1) / 2.0 + (n & 1));
            auto put = [&](int idx, double ang) { h3[idx] = {std::cos(ang), std::sin(ang)}; };
            put(n, th / 2);
            put(16 + n, th / 4);
            for (int b = 0; b < 2; ++b) put(32 + 16 * b + n, th / 8 + PI * b / 4);
            for (int b = 0; b < 4; ++b) put(64 + 16 * b + n, th / 16 + PI * ((b >> 1) / 8.0 + (b & 1) / 4.0));
            for (int p = 0; p < 8; ++p)
                for (int b8 = 0; b8 < 2; ++b8)
                    put(128 + 32 * p + n + 16 * b8, th / 32 + PI * ((p >> 2) / 16.0 + ((p >> 1) & 1) / 8.0 + (p & 1) / 4.0) +
                                                        PI / 2 * b8);
        }
        // Pw256Regs at lane 16 k0 + .. (powers over c), 4 (4 k0 + e) + .. (over g), 16 k0 + 4 e + p (over h)
        cplx* h4 = h3 + 384;
        for (int l = 0; l < 64; ++l) {
            const int k0 = l >> 4, k = k0 + 4 * ((l >> 2) & 3), p = l & 3;
            // exp(i pi / 512 (1 - 4 k) m)
            auto put = [&](int idx, int kk, int m) {
                const double ang = PI * (double)(((1 - 4 * kk) * m) % 1024) / 512.0;
                h4[idx * 64 + l] = {std::cos(ang), std::sin(ang)};
            };
            put(0, k0, 16);
            put(1, k0, 32);
            put(2, k, 4);
            put(3, k, 8);
            put(4, k + 16 * p, 1);
            put(5, k + 16 * p, 2);
        }
        int rc = dmalloc((void**)&d_buf, h.size() * sizeof(cplx));
        if (rc) return rc;
        rc = hipcheck(hipMemcpy(d_buf, h.data(), h.size() * sizeof(cplx), hipMemcpyHostToDevice), "tables");
        if (rc) return rc;
        T.p1t = d_buf;
        T.p2 = d_buf + 512;
        T.rot = d_buf + 1024;
        T.two = d_buf + 1024 + 2 * N;
        T.pair = T.two + 1024;
        T.pw = T.pair + 384;
        return TFHE_OK;
    }
    void release() {
        if (d_buf) (void)hipFree(d_buf);
        d_buf = nullptr;
    }
};

// Twiddle tables of the 4-wave N = 2048 FFT (fft1024.hpp): p1t, p2, p3 [4][64],
// tr [4][4][64], rot [2N], pw [10][16]; 6048 complex values.
struct DeviceTables1024 {
    FFT1024Tables T{};
    cplx* d_buf = nullptr;
    // rounded: fft_tables.hpp
    int init(bool rounded = false) {
        const std::vector<TableValue> h = fft1024_tables(rounded);
        static_assert(sizeof(TableValue) == sizeof(cplx), "the tables' values are copied as they are");
        int rc = dmalloc((void**)&d_buf, h.size() * sizeof(cplx));
        if (rc) return rc;
        rc = hipcheck(hipMemcpy(d_buf, h.data(), h.size() * sizeof(cplx), hipMemcpyHostToDevice), "tables1024");
        if (rc) return rc;
        T.p1t = d_buf;
        T.p2 = d_buf + 256;
        T.p3 = d_buf + 512;
        T.tr = d_buf + 768;
        T.rot = d_buf + 1792;
        T.pw = d_buf + 1792 + 4096;
        return TFHE_OK;
    }
    void release() {
        if (d_buf) (void)hipFree(d_buf);
        d_buf = nullptr;
    }
};

// The same tables rounded to FP32 (the split-precision product).
struct DeviceTables1024F {
    FFT1024TablesF T{};
    cplxf* d_buf = nullptr;
    int init() {
        const std::vector<TableValue> h = fft1024_tables(false);
        std::vector<cplxf> f(h.size());
        for (size_t k = 0; k < h.size(); ++k) f[k] = {(float)h[k].re, (float)h[k].im};
        int rc = dmalloc((void**)&d_buf, f.size() * sizeof(cplxf));
        if (rc) return rc;
        rc = hipcheck(hipMemcpy(d_buf, f.data(), f.size() * sizeof(cplxf), hipMemcpyHostToDevice), "tables1024f");
        if (rc) return rc;
        T.p1t = d_buf;
        T.p2 = d_buf + 256;
        T.p3 = d_buf + 512;
        T.tr = d_buf + 768;
        T.rot = d_buf + 1792;
        T.pw = d_buf + 1792 + 4096;
        return TFHE_OK;
    }
    void release() {
        if (d_buf) (void)hipFree(d_buf);
        d_buf = nullptr;
    }
};

// Process-lifetime twiddle tables for the stateless entry points, one set per
// device (tables in one device's memory are not read from another), each built
// once under a lock.
constexpr int kMaxDevices = 64;
template <class Tables, class Init>
int per_device_tables(Tables*& out, Init init) {
    static std::mutex mu;
    static Tables tables[kMaxDevices];
    int dev = 0;
    int rc = hipcheck(hipGetDevice(&dev), "get device");
    if (rc) return rc;
    if (dev < 0 || dev >= kMaxDevices) return fail(TFHE_E_PARAM, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!tables[dev].d_buf) {
        rc = init(tables[dev]);
        if (rc) return rc;
    }
    out = &tables[dev];
    return TFHE_OK;
}

// Batched gate bootstrap with the scratch passed in: lweN holds [batch][N+1] u32 (blind-rotation
// outputs), ks_at [N][ks_bpad(batch)] u32 (key-switch digits); cap is the largest batch they hold.
int gate_eval_with_scratch(tfhe_gate_ctx* c, int gate, const uint32_t* d_ct1, const uint32_t* d_ct2, uint32_t batch,
                           uint32_t cap, uint32_t* d_out, uint32_t* lweN, uint32_t* ks_at, void* stream);

// Looks up the no-allocation entry point's device array on the current GPU (once per device).
int noalloc_prepare_current_device();

}  // namespace tfhe
