"""The kernel forms that a launch's size chooses, at the sizes where one begins or a workgroup is
partly filled: the same words as the other form's, and the oracle's on sampled inputs."""
import numpy as np
import pytest

import oracle as O
from conftest import from_dev, to_dev

pytestmark = pytest.mark.gpu

SEED = 21


@pytest.fixture(scope="module")
def gkeys():
    return O.GateKeys(3)


@pytest.fixture(scope="module")
def gctx(gpu, gkeys):
    import tfhe_amd
    c = tfhe_amd.GateContext(max_batch=2048)
    c.set_keys(gkeys.bsk, gkeys.ksk)
    yield c
    c.close()


@pytest.fixture(scope="module")
def okeys():
    return O.CbsKeys(SEED)


@pytest.fixture(scope="module")
def ctx(gpu, okeys):
    import tfhe_amd
    c = tfhe_amd.CbsContext(max_blocks=9)
    c.keygen(okeys.s, SEED)
    yield c
    c.close()


def _rand(shape, seed, bits=32):
    t = np.uint32 if bits == 32 else np.uint64
    return np.random.default_rng(seed).integers(0, 2 ** bits, shape, dtype=np.uint64).astype(t)


@pytest.mark.parametrize("count", [1, 31, 33, 255, 256, 257, 481, 511, 512, 513, 1100])
def test_pfks_counts(ctx, okeys, count):
    """Lookup PFKS: 32 inputs per wave, 256 (up to 256 inputs) or 512 per workgroup.  Five inputs
    (every digit value, the wrap of the rounding, zero, random ones) repeated over the launch:
    each row equals the oracle's."""
    import torch
    base = _rand((5, 2049), 12, 64)
    base[0, :64] = np.uint64(2 ** 64 - 2 ** 31 + 5)
    base[1, :16] = np.array([(v * 0x11111111) << 32 for v in range(16)], np.uint64)
    base[2] = 0
    pick = np.arange(count) * 7 % 5
    d_in = torch.from_numpy(base[pick].view(np.int64).copy()).to("cuda")
    for u in (0, 1):
        d_out = torch.full((count + 1, 4096), 7, dtype=torch.int32, device="cuda")
        ctx.pfks_batch(u, d_in, count, 4096, d_out)
        torch.cuda.synchronize()
        got = from_dev(d_out)
        want = np.stack([okeys.pfks(u, base[j]) for j in range(5)])
        assert np.array_equal(got[:count], want[pick]), u
        assert (got[count] == 7).all()


@pytest.mark.parametrize("func", [False, True])
def test_gate_forms(gctx, gkeys, func):
    """768 gates (three rounds of one ciphertext per workgroup on 256 CUs) and 769 (four one-wave
    ciphertexts per workgroup, the last alone): equal rows, and a ciphertext without a mask."""
    import torch
    n1 = gkeys.p.n + 1
    c1, c2 = _rand((769, n1), 1), _rand((769, n1), 2)
    c1[5] = c2[5] = 0
    rows = {}
    for count in (1, 768, 769):
        first = 5 if count == 1 else 0
        d1, d2 = to_dev(c1[first:first + count]), to_dev(c2[first:first + count])
        d_out = torch.empty((count, n1), dtype=torch.int32, device="cuda")
        if func:
            lut = np.repeat(np.arange(4, dtype=np.uint32) * 256, 256)
            gctx.eval_func(to_dev(c1[first:first + count] & 1023), 1024, lut, d_out)
        else:
            gctx.eval_batch(O.XOR, d1, d2, d_out)
        torch.cuda.synchronize()
        rows[count] = from_dev(d_out)
    assert np.array_equal(rows[768], rows[769][:768])
    assert np.array_equal(rows[1][0], rows[768][5])
    if not func:
        for k in (5, 768):
            want, _ = gkeys.bootstrap(O.XOR, c1[k], c2[k])
            assert np.array_equal(rows[769][k], want), k


@pytest.mark.parametrize("count", [1, 128, 129, 256, 257])
def test_keyswitch_slices(gctx, gkeys, count):
    """N = 1024 key switch with one, two and three ciphertext groups."""
    import torch
    lwe = _rand((3, gkeys.p.N + 1), 9)
    pick = np.arange(count) % 3
    d_out = torch.empty((count, gkeys.p.n + 1), dtype=torch.int32, device="cuda")
    gctx.keyswitch_batch(to_dev(lwe[pick]), d_out)
    torch.cuda.synchronize()
    want = np.stack([O.keyswitch32(gkeys, lwe[j]) for j in range(3)])
    assert np.array_equal(from_dev(d_out), want[pick])


@pytest.mark.parametrize("form", ["exact", "one_bit", "two_bits", "htss"])
def test_pbs_pairs_and_odd_batches(gpu, okeys, form):
    """Launches above 256 inputs run two ciphertexts per workgroup (one-bit one-product: one); an
    odd batch's last workgroup stores one.  Rows of 257 and 258 inputs agree, the row past the end
    is untouched, and a ciphertext without a mask bootstraps as in a launch of its own (the
    one-product forms sum in another order there, so only the exact ones compare words)."""
    import torch
    import tfhe_amd
    params = {"exact": {}, "one_bit": {"pbs_approx": 1}, "two_bits": {"pbs_approx": 1, "pbs_multibit": 2},
              "htss": {"lwe_to_rgsw": 1}}[form]
    c = tfhe_amd.CbsContext(max_blocks=3, params=tfhe_amd.cbs_params(**params))
    c.keygen(okeys.s, SEED)
    cts = _rand((258, okeys.p.n + 1), 3)
    cts[1, :-1] = 0
    cts[2, :-1] = 0
    cts[2, 7] = 1 << 29
    rows = {}
    for count in (257, 258):
        if form == "htss":
            d_out = torch.full((count + 1, 4, 2, 2048), 7, dtype=torch.int32, device="cuda")
            c.cbs_batch(to_dev(cts[:count]), d_out[:count])
        else:
            d_out = torch.full((count + 1, 2, 2049), 7, dtype=torch.int64, device="cuda")
            c.pbs_batch(to_dev(cts[:count]), d_out[:count])
        torch.cuda.synchronize()
        rows[count] = d_out.cpu().numpy()
        assert (rows[count][count] == 7).all()
    assert np.array_equal(rows[257][:257], rows[258][:257])
    d_one = torch.empty_like(d_out[:3])
    (c.cbs_batch if form == "htss" else c.pbs_batch)(to_dev(cts[:3]), d_one)
    torch.cuda.synchronize()
    if form in ("exact", "htss"):
        assert np.array_equal(d_one.cpu().numpy(), rows[257][:3])
    c.close()


@pytest.mark.parametrize("params", [{}, {"pbs_approx": 1, "pbs_multibit": 2}], ids=["exact", "two_bits"])
def test_pbs_small_launches(gpu, okeys, params):
    """Up to 64 inputs run 16 to an XCD, more are dealt to all of them: a prefix of a launch of 128
    gives its rows, and nothing past it is written."""
    import torch
    import tfhe_amd
    c = tfhe_amd.CbsContext(max_blocks=1, params=tfhe_amd.cbs_params(**params))
    c.keygen(okeys.s, SEED)
    d_cts = to_dev(_rand((128, okeys.p.n + 1), 4))
    d_all = torch.empty((128, 2, 2049), dtype=torch.int64, device="cuda")
    c.pbs_batch(d_cts, d_all)
    for count in (1, 15, 17, 33, 50, 64, 65):
        d_out = torch.full((count + 1, 2, 2049), 7, dtype=torch.int64, device="cuda")
        c.pbs_batch(d_cts[:count].contiguous(), d_out[:count])
        torch.cuda.synchronize()
        assert torch.equal(d_out[:count], d_all[:count]), count
        assert bool((d_out[count] == 7).all())
    c.close()


def test_pfks_linear_counts(gpu, okeys):
    """Linear PFKS: 128-input tiles up to 256 inputs, 256-input tiles staged through LDS above; the
    rows of each launch equal those of launches of 64, and the oracle's on the first and last."""
    import torch
    import tfhe_amd
    c = tfhe_amd.CbsContext(max_blocks=3, params=tfhe_amd.cbs_params(pfks_linear=1))
    c.keygen(okeys.s, SEED)
    lwe = _rand((600, 2049), 6, 64)
    d_in = torch.from_numpy(lwe.view(np.int64).copy()).to("cuda")
    for u in (0, 1):
        d_ref = torch.empty((600, 4096), dtype=torch.int32, device="cuda")
        for k in range(0, 600, 64):
            m = min(64, 600 - k)
            c.pfks_batch(u, d_in[k:k + m].contiguous(), m, 4096, d_ref[k:k + m])
        for count in (1, 128, 255, 256, 257, 511, 513, 600):
            d_out = torch.full((count + 1, 4096), 7, dtype=torch.int32, device="cuda")
            c.pfks_batch(u, d_in[:count].contiguous(), count, 4096, d_out)
            torch.cuda.synchronize()
            assert torch.equal(d_out[:count], d_ref[:count]), (u, count)
            assert bool((d_out[count] == 7).all())
        for k in (0, 599):
            assert np.array_equal(from_dev(d_ref)[k], okeys.pfks_linear(u, lwe[k])), (u, k)
    c.close()


@pytest.mark.parametrize("count", [640, 767, 768, 769, 1025, 1280, 1281])
def test_pfks_rest_launch(ctx, okeys, count):
    """Lookup PFKS of whole groups of 512 inputs and a rest: up to 256 of it run as a launch of their
    own, more in the groups' launch; each row equals the oracle's, at a stride wider than a row."""
    import torch
    base = _rand((5, 2049), 15, 64)
    pick = np.arange(count) * 3 % 5
    d_in = torch.from_numpy(base[pick].view(np.int64).copy()).to("cuda")
    for u in (0, 1):
        d_out = torch.full((count + 1, 4100), 7, dtype=torch.int32, device="cuda")
        ctx.pfks_batch(u, d_in, count, 4100, d_out)
        torch.cuda.synchronize()
        got = from_dev(d_out)
        want = np.stack([okeys.pfks(u, base[j]) for j in range(5)])
        assert np.array_equal(got[:count, :4096], want[pick]), u
        assert (got[count] == 7).all() and (got[:, 4096:] == 7).all()


@pytest.mark.parametrize("count", [257, 320, 384, 385, 600])
def test_cbs_rest_launch(ctx, okeys, count):
    """The same with both functions in a launch (2 count PFKS inputs of a circuit bootstrap batch):
    the rows of batches of 64."""
    import torch
    d_in = to_dev(_rand((count, okeys.p.n + 1), 16))
    d_out = torch.full((count + 1, 4, 2, 2048), 7, dtype=torch.int32, device="cuda")
    ctx.cbs_batch(d_in, d_out[:count])
    d_ref = torch.empty((count, 4, 2, 2048), dtype=torch.int32, device="cuda")
    for k in range(0, count, 64):
        ctx.cbs_batch(d_in[k:k + 64].contiguous(), d_ref[k:k + 64])
    torch.cuda.synchronize()
    assert torch.equal(d_out[:count], d_ref)
    assert bool((d_out[count] == 7).all())


def _least_ms(fn, passes=8):
    import torch
    fn()
    best = float("inf")
    for _ in range(passes):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        fn()
        t1.record()
        torch.cuda.synchronize()
        best = min(best, t0.elapsed_time(t1))
    return best


def test_pfks_rest_is_not_a_whole_group(ctx):
    """600 lookup PFKS take no longer than launches of 512 and 88 do (1.35 times as long when the 88
    waited in a whole group's time); 1.15 allows for what two timings differ by."""
    import torch
    d_in = torch.from_numpy(_rand((600, 2049), 17, 64).view(np.int64).copy()).to("cuda")
    d_out = torch.empty((600, 4096), dtype=torch.int32, device="cuda")
    whole = _least_ms(lambda: ctx.pfks_batch(1, d_in, 600, 4096, d_out))
    parts = (_least_ms(lambda: ctx.pfks_batch(1, d_in, 512, 4096, d_out)) +
             _least_ms(lambda: ctx.pfks_batch(1, d_in[512:], 88, 4096, d_out[512:])))
    assert whole < 1.15 * parts, (whole, parts)


def test_pfks_linear_one_function(gpu, okeys):
    """Linear PFKS of one function: 128-input tiles up to 512 inputs, where one round of workgroups
    holds them.  The rows of 385, 512 and 513 inputs are those of launches of 64, and 300
    inputs take about what 256 do (1.27 times as long in staged 256-input tiles, which leave half of
    the chip idle there; 1.15 allows for what two timings differ by)."""
    import torch
    import tfhe_amd
    c = tfhe_amd.CbsContext(max_blocks=3, params=tfhe_amd.cbs_params(pfks_linear=1))
    c.keygen(okeys.s, SEED)
    d_in = torch.from_numpy(_rand((513, 2049), 18, 64).view(np.int64).copy()).to("cuda")
    d_out = torch.full((514, 4096), 7, dtype=torch.int32, device="cuda")
    for u in (0, 1):
        d_ref = torch.empty((513, 4096), dtype=torch.int32, device="cuda")
        for k in range(0, 513, 64):
            m = min(64, 513 - k)
            c.pfks_batch(u, d_in[k:k + m].contiguous(), m, 4096, d_ref[k:k + m])
        for count in (385, 512, 513):
            d_out.fill_(7)
            c.pfks_batch(u, d_in, count, 4096, d_out)
            torch.cuda.synchronize()
            assert torch.equal(d_out[:count], d_ref[:count]), (u, count)
            assert bool((d_out[count] == 7).all())
    t256 = _least_ms(lambda: c.pfks_batch(1, d_in, 256, 4096, d_out), 20)
    t300 = _least_ms(lambda: c.pfks_batch(1, d_in, 300, 4096, d_out), 20)
    assert t300 < 1.15 * t256, (t300, t256)
    c.close()


def _phase64(K2, r):
    return O.rlwe_phase64(K2, np.ascontiguousarray(r).reshape(-1)).astype(np.uint64)


@pytest.mark.parametrize("form", ["exact", "one_bit", "two_bits", "htss"])
def test_many_lut_forms(gpu, okeys, form):
    """A caller's test polynomial in the launches that two ciphertexts share (257 and 258 inputs) and in
    small ones, at bitwidths 0 and 1: rotations are odd and even at 0, so the factors of a
    lane's frequencies differ, and even at 1.  Inputs: random words, a zero mask, one rotating key
    bit.  Exact forms: the oracle's words, of the last odd input too.  One-product forms: every
    coefficient's phase within 2^40 of 2^64 of the exact oracle's (both carry the PBS noise, about
    2^36 rms)."""
    import os
    from concurrent.futures import ThreadPoolExecutor
    import torch
    import tfhe_amd
    params = {"exact": {}, "one_bit": {"pbs_approx": 1}, "two_bits": {"pbs_approx": 1, "pbs_multibit": 2},
              "htss": {"lwe_to_rgsw": 1}}[form]
    keys = O.CbsKeys(SEED, p=O.cbs_params_htss()) if form == "htss" else okeys
    mb = 2 if form == "two_bits" else 1
    if mb == 2:
        keys.bsk_mb2_fourier()
    c = tfhe_amd.CbsContext(max_blocks=3, params=tfhe_amd.cbs_params(**params))
    c.keygen(keys.s, SEED)
    cts = _rand((258, keys.p.n + 1), 19)
    cts[1, :-1] = 0
    cts[2, :-1] = 0
    cts[2, 7] = 0x2345678
    cts[255] = cts[1]
    lut = _rand(keys.p.N, 20, 64)
    d_lut = torch.from_numpy(lut.view(np.int64).copy()).to("cuda")
    rows = [0, 1, 2, 3, 255, 256, 257]
    for bw in (0, 1):
        with ThreadPoolExecutor(max(1, min(16, os.cpu_count() or 1))) as pool:
            want = dict(zip(rows, pool.map(lambda k: keys.bootstrap_many_lut(cts[k], lut, bw, mb=mb), rows)))
        for count in (4, 257, 258):
            d_out = torch.full((count + 1, 2, keys.p.N), 7, dtype=torch.int64, device="cuda")
            c.bootstrap_many_lut(to_dev(cts[:count]), d_lut, bw, d_out[:count])
            torch.cuda.synchronize()
            got = from_dev(d_out, np.uint64)
            assert (got[count] == 7).all()
            for k in rows:
                if k >= count:
                    continue
                exact, err = want[k]
                assert err < 0.25
                if form in ("exact", "htss") or k in (1, 255):  # a zero mask: no products
                    assert np.array_equal(got[k], exact), (bw, count, k)
                else:
                    d = (_phase64(keys.K2, got[k]) - _phase64(keys.K2, exact)).view(np.int64)
                    assert np.abs(d).max() < 2 ** 40, (bw, count, k)
    c.close()


@pytest.mark.parametrize("form", ["one_bit", "two_bits"])
def test_one_product_forms_agree(gpu, okeys, form):
    """One key bit per step is one kernel at every size: 3 inputs and 257 give the same words.  Two key
    bits: two ciphertexts per workgroup (form 0) and one split over 8 waves (form 2) sum in
    another order; a zero mask (no products) gives the same words, and one rotating key bit a phase
    within 2^30 of 2^64 (the first step's rounding is 2^25 rms).  The last odd input of 257 agrees
    with the oracle's exact bootstrap within 2^40."""
    import torch
    import tfhe_amd
    mb = 2 if form == "two_bits" else 1
    c = tfhe_amd.CbsContext(max_blocks=3, params=tfhe_amd.cbs_params(pbs_approx=1, pbs_multibit=mb))
    c.keygen(okeys.s, SEED)
    cts = _rand((257, okeys.p.n + 1), 21)
    cts[:3, :-1] = 0
    cts[1, 7] = 1 << 29
    cts[2, 400] = 0x9abcdef0

    def run(count):
        d_out = torch.full((count + 1, 2, 2049), 7, dtype=torch.int64, device="cuda")
        c.pbs_batch(to_dev(cts[:count]), d_out[:count])
        torch.cuda.synchronize()
        assert bool((d_out[count] == 7).all())
        return from_dev(d_out, np.uint64)[:count]

    large = run(257)
    K = okeys.K2.astype(np.int64).astype(np.uint64)

    def apart(a, b):  # phases of two outputs, both levels
        d = (a[:, -1] - (a[:, :-1] * K).sum(1, dtype=np.uint64)) - (b[:, -1] - (b[:, :-1] * K).sum(1, dtype=np.uint64))
        return int(np.abs(d.view(np.int64)).max())

    if mb == 1:
        assert np.array_equal(run(3), large[:3])
        assert np.array_equal(run(256), large[:256])
    else:
        for count in (3, 256):
            pinned = {}
            for f in (0, 2):
                c.set_pbs_form(count, f)
                pinned[f] = run(count)
            c.set_pbs_form(count, -1)
            assert np.array_equal(run(count), pinned[2])  # the size rule's choice
            assert np.array_equal(pinned[0], large[:count])
            assert np.array_equal(pinned[2][0], large[0])
            for k in (1, 2):
                assert apart(pinned[2][k], large[k]) < 2 ** 30, (count, k)
            for k in range(3, count):
                assert apart(pinned[2][k], large[k]) < 2 ** 40, (count, k)
    want, err = okeys.pbs_mb2(cts[256]) if mb == 2 else okeys.pbs(cts[256])
    assert err < 0.25
    assert apart(large[256], want) < 2 ** 40
    c.close()


@pytest.mark.parametrize("params,forms", [({}, (0, 1)), ({"pbs_approx": 1}, (1,)),
                                          ({"pbs_approx": 1, "pbs_multibit": 2}, (0, 2)),
                                          ({"pbs_approx": 1, "pbs_multibit": 3}, (1, 2, 4))],
                         ids=["exact", "one_bit", "two_bits", "auto"])
def test_autotune_reports_each_kernel_by_one_number(gpu, okeys, params, forms):
    """The tuner times each PBS kernel once: the choices of 1, 3 and 5 blocks (5: a full round and a
    rest) name one of the context's kernels, never an alias, and the aliases stay accepted."""
    import tfhe_amd
    c = tfhe_amd.CbsContext(max_blocks=5, params=tfhe_amd.cbs_params(**params))
    c.keygen(okeys.s, SEED)
    for blocks in (1, 3, 5):
        chosen = c.autotune(blocks)["pbs_form"]
        assert all(f in forms for f in chosen[blocks < 5:]), (blocks, chosen)
    for f in range(max(forms) + 1):
        c.set_pbs_form(77, f)
    with pytest.raises(tfhe_amd.TfheError):
        c.set_pbs_form(77, 5 if params.get("pbs_multibit") == 3 else max(forms) + 1)
    c.close()
