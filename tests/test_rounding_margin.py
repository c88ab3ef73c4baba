"""How far the exact forms' FP64 products end from the integers they are rounded to.

The GPU's exact bootstraps take (X^m - 1) sum_r d_r K_r, signed digits times signed 32-bit key
words, through an FP64 transform and round once: the words are exact while the computed value lies
within 1/2 of the integer.  Here the same transforms run in numpy (radix-4 steps with the twiddles
fused, the cross-wave step of four 256-point transforms, the factor w^(m (1 - 4k)) - 1 before
the inverse; for N = 1024 the binary splitting of x^512 - i), against the exact integer.  numpy
has no fused multiply-add, so every product is rounded once more than on the GPU."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "gpu-circuitbootstrapping-aestransciphering_amd", "csrc")


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    """The library's own N = 2048 tables (fft_tables.hpp): {rounded: complex values in device order}."""
    exe = str(tmp_path_factory.mktemp("tables") / "dump")
    src = ('#include <cstdio>\n#include "fft_tables.hpp"\nint main(int n, char**) {\n'
           'const auto h = tfhe::fft1024_tables(n > 1);\n'
           'return fwrite(h.data(), sizeof h[0], h.size(), stdout) == h.size() ? 0 : 1; }\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", CSRC, "-o", exe, "-x", "c++", "-"],
                   input=src, text=True, check=True, timeout=120)
    return {bool(args): np.frombuffer(subprocess.run([exe] + args, capture_output=True, check=True).stdout,
                                      np.complex128) for args in ([], ["rounded"])}


def _w(x):
    """exp(i pi x)"""
    return np.exp(1j * np.pi * np.asarray(x, np.float64))


def _dft4(x, sign):
    a0, a1, b0, b1 = x[0] + x[2], x[0] - x[2], x[1] + x[3], sign * 1j * (x[1] - x[3])
    return [a0 + b0, a1 + b1, a0 - b0, a1 - b1]


def _dft4_pw(x, w1, w2, sign):
    """radix-4 of x[j] w1^j, w2 = w1^2, as the kernels fuse it"""
    e = x[0] + w2 * x[2]
    f = 2 * x[0] - e
    g = x[1] + w2 * x[3]
    h = 2 * x[1] - g
    y0, y1 = e + w1 * g, f + sign * 1j * w1 * h
    return [y0, y1, 2 * e - y0, 2 * f - y1]


R4 = np.arange(4)


class Fft2048:
    """Transform of the N = 2048 forms: point 4 b + r of wave r, b = 64 a + 16 c + 4 g + h;
    frequency k + 256 q of wave k's top bits, k = k0 + 4 e + 16 p + 64 s."""
    N = 2048

    def __init__(self, tab):
        k = np.arange(256)
        lane = 16 * (k & 3) + 4 * ((k >> 2) & 3) + ((k >> 4) & 3)
        p1t, p2 = tab[:256].reshape(4, 64), tab[256:512].reshape(4, 64)
        self.p1t = p1t.T.reshape(4, 4, 4, 4)                                 # [c][g][h][k0], b = 16 c + 4 g + h
        self.w64 = p2[1:3, :16].reshape(2, 4, 4, 1)                          # W64^d, W64^2d at [g][h]
        self.tr = tab[768:1792].reshape(4, 4, 64)[:, k >> 6, lane]           # T_r[k]
        self.rot = tab[1792:5888]
        self.pw = tab[5888:].reshape(10, 4, 4)                               # [power][k0][e]
        self.ek = (1 - 4 * (k[None] + 256 * R4[:, None])) % 4096             # [q][k]

    def _fwd256(self, x):  # [.., b] -> [.., k]
        x = x.reshape(x.shape[:-1] + (4, 4, 4, 4))  # a, c, g, h
        x = np.stack(_dft4_pw([x[..., a, :, :, :] for a in range(4)], _w(4 / 32), _w(8 / 32), -1), -4)  # k0, c, g, h
        k0 = R4[:, None, None]
        x = np.stack(_dft4_pw([x[..., :, c, :, :] for c in range(4)], _w((1 - 4 * k0) / 32), _w((2 - 8 * k0) / 32),
                              -1), -3)  # k0, e, g, h
        x = np.stack(_dft4_pw([x[..., g, :] for g in range(4)], self.pw[0][:, :, None], self.pw[1][:, :, None], -1), -2)
        x = np.stack(_dft4_pw([x[..., h] for h in range(4)], np.moveaxis(self.pw[2::2], 0, -1),
                              np.moveaxis(self.pw[3::2], 0, -1), -1), -1)  # k0, e, p, s
        return np.moveaxis(x, (-4, -3, -2, -1), (-1, -2, -3, -4)).reshape(x.shape[:-4] + (256,))

    def _inv256(self, x):  # [.., k] -> 256 x [.., b]
        x = x.reshape(x.shape[:-1] + (4, 4, 4, 4))  # s, p, e, k0
        x = np.stack(_dft4([x[..., s, :, :, :] for s in range(4)], 1), -4)  # h, p, e, k0
        h = R4[:, None, None]
        x = np.stack(_dft4_pw([x[..., :, p, :, :] for p in range(4)], _w(4 * h / 32), _w(8 * h / 32), 1), -4)
        # g, h, e, k0
        w64 = np.conj(self.w64)
        x = np.stack(_dft4_pw([x[..., e, :] for e in range(4)], w64[0], w64[1], 1), -4)  # c, g, h, k0
        x = x * np.conj(self.p1t)
        x = np.stack(_dft4([x[..., k0] for k0 in range(4)], 1), -4)  # a, c, g, h
        return (x * np.conj(_w(R4 / 8))[:, None, None, None]).reshape(x.shape[:-4] + (256,))

    def forward(self, p):  # [.., N] -> [.., q, k]
        z = p[..., :1024] + 1j * p[..., 1024:]
        y = self._fwd256(np.moveaxis(z.reshape(z.shape[:-1] + (256, 4)), -1, -2))
        return np.stack(_dft4_pw([y[..., r, :] for r in range(4)], self.tr[1], self.tr[2], -1), -2)

    def factor(self, m):
        return self.rot[m * self.ek % 4096] - 1.0

    def inverse(self, x):
        y = np.stack(_dft4([x[..., q, :] for q in range(4)], 1), -2) * np.conj(self.tr)
        z = np.moveaxis(self._inv256(y), -2, -1).reshape(x.shape[:-2] + (1024,)) / 1024
        return np.concatenate([z.real, z.imag], -1)


class Fft1024:
    """The N = 1024 pair transform: x^512 - i split nine times, leaf order."""
    N = 1024

    def __init__(self):
        th = np.array([0.5])
        self.half = []
        for _ in range(9):
            self.half.append(th / 2)
            th = np.stack([th / 2, th / 2 + 1], -1).reshape(-1)
        self.e = np.rint(th * 1024).astype(np.int64) % 2048  # roots w^e
        self.rot = _w(np.arange(2048) / 1024)

    def forward(self, p):
        x = (p[..., :512] + 1j * p[..., 512:])[..., None, :]
        for th in self.half:
            m = x.shape[-1] // 2
            lo, hi = x[..., :m], x[..., m:]
            s = lo + _w(th)[:, None] * hi
            x = np.stack([s, 2 * lo - s], -2).reshape(x.shape[:-2] + (-1, m))
        return x[..., 0]

    def factor(self, m):
        """w^(m e) from one table value and the powers of w^(64 m), w^(128 m), w^(256 m), e = e0 + their
        multiples, with the inverse's 1 / 512"""
        e0 = self.e & ~(64 + 128 + 256)
        z = self.rot[m * e0 % 2048] / 512
        for b in (64, 128, 256):
            z = np.where(self.e & b, z * self.rot[b * m % 2048], z)
        return z - 1 / 512

    def inverse(self, x):
        x = x[..., None]
        for th in reversed(self.half):
            x = x.reshape(x.shape[:-2] + (-1, 2, x.shape[-1]))
            p, q = x[..., 0, :], x[..., 1, :]
            x = np.concatenate([p + q, (p - q) * np.conj(_w(th))[:, None]], -1)
        return np.concatenate([x[..., 0, :].real, x[..., 0, :].imag], -1)


def _negacyclic(d, K):
    """sum over rows of d * K mod X^N + 1 as exact integers: K in 16-bit halves, so that the FP64
    convolutions (below 2^40) are off by far less than 1/2"""
    N = d.shape[-1]
    t = _w(np.arange(N) / N)
    D = np.fft.fft(d * t)
    out = np.zeros(N, np.int64)
    for part, shift in ((K >> 16, 16), (K & 0xFFFF, 0)):
        y = np.fft.ifft((D * np.fft.fft(part * t)).sum(0)) * np.conj(t)
        out += np.rint(y.real).astype(np.int64) << shift
    return out


def _monic(t, m):  # (X^m - 1) t
    N = t.size
    k = np.arange(N) - m
    return np.where((k // N) % 2 != 0, -t[k % N], t[k % N]) - t


def _distances(F, rows, digits, steps, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(steps):
        d = digits(rng, (rows, F.N))
        K = rng.integers(-2 ** 31, 2 ** 31, (rows, F.N))
        m = int(rng.integers(1, 2 * F.N))
        y = (F.forward(d.astype(np.float64)) * F.forward(K.astype(np.float64))).sum(0) * F.factor(m)
        exact = _monic(_negacyclic(d, K), m)
        assert np.abs(exact).max() < 2 ** 51  # the rounding by 1.5 * 2^52 holds
        out.append(F.inverse(y) - exact)
    return np.abs(np.concatenate(out))


def _uniform(half):
    return lambda rng, shape: rng.integers(-half, half, shape)


def _check(name, e):
    """The largest distance stays below 1/4, half of what rounding allows, and the rms below a
    tenth of 1/2: the distances are sums of many independent roundings, so ten times the rms is not
    met in any number of bootstraps."""
    rms = np.sqrt(np.mean(e ** 2))
    print(f"{name}: distance from the integer rms {rms:.4f}, largest {e.max():.3f} of {e.size}")
    assert e.max() < 0.25
    assert rms < 0.05


@pytest.mark.parametrize("name,rows,digits,steps", [
    ("2^9 x 4", 8, _uniform(256), 40),
    ("2^10 x 4 (HomTrace + SchemeSwitch)", 8, _uniform(512), 40),
    # a caller's polynomial as the first step meets it: no mask, every digit the largest
    ("2^10 x 4, largest digits of one sign", 4, lambda rng, shape: np.full(shape, -512), 20),
    ("2^10 x 4, largest digits", 4, lambda rng, shape: 1024 * rng.integers(0, 2, shape) - 512, 20),
], ids=["pbs", "pbs_htss", "largest_one_sign", "largest"])
def test_pbs_products_round_to_their_integers(tables, name, rows, digits, steps):
    """The exact PBS with the tables its contexts hold."""
    _check(name, _distances(Fft2048(tables[True]), rows, digits, steps, 3))


def test_gate_products_round_to_their_integers():
    _check("gate, 2^7 x 3", _distances(Fft1024(), 6, _uniform(64), 40, 3))


def test_tables_are_rounded_once(tables):
    """Both table sets against the same angles in long double; the exact contexts' within half a
    unit in the last place of 1 (1.1e-16), the one-product contexts' within ten."""
    pi = np.longdouble("3.14159265358979323846264338327950288")

    def w(num, den):
        a = pi * (np.asarray(num) % (2 * den)).astype(np.longdouble) / den
        return np.cos(a), np.sin(a)

    l, k, r4 = np.arange(64), np.arange(16), R4[:, None]
    kk = (l >> 4) + 4 * ((l >> 2) & 3) + 16 * (l & 3) + 64 * R4[:, None]
    kp = (1 - 4 * ((k >> 2) + 4 * (k & 3) + 16 * R4[:, None]))[:, None, :] * np.array([1, 2])[:, None]
    want = [w(4 * l - 16 * l * r4, 2048), w(-2 * (l & 15) * r4, 64), w(-2 * (l & 3) * r4, 16),
            w(R4[:, None, None] * (1 - 4 * kk), 2048), w(np.arange(4096), 2048),
            w((1 - 4 * ((k >> 2) + 4 * (k & 3))) * np.array([[4], [8]]), 512), w(kp, 512)]
    re, im = (np.concatenate([v[i].reshape(-1) for v in want]) for i in (0, 1))
    for rounded, bound in ((True, 2.0 ** -53 * 1.01), (False, 10 * 2.0 ** -53)):
        t = tables[rounded]
        assert t.size == re.size
        assert max(np.abs(t.real - re).max(), np.abs(t.imag - im).max()) <= bound, rounded
