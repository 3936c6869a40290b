"""EDEN Lloyd-Max quantiser / THC uniform quantiser kernels: bit-exact against the oracle; the host mirrors
against the reference's own outputs (tests/golden/eden_golden.npz) and the reference's torch op chains."""
import math
import os

import numpy as np
import pytest
import torch

from helpers import to_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "eden_golden.npz"))


def _tables(nbits):
    return (torch.from_numpy(GOLD["centroids_%d" % nbits]).to(DEV), torch.from_numpy(GOLD["boundaries_%d" % nbits]).to(DEV))


@pytest.mark.parametrize("nbits", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n", [32, 1024, 4096 * 3 + 64, 1 << 20])
def test_eden_quantize_bit_exact(capi, oracle, nbits, n):
    g = torch.Generator().manual_seed(n + nbits)
    x = torch.randn(n, generator=g) * 3e-3
    if n > 64:
        x[5] = 0.0
        x[7:40] *= 50.0                       # outliers beyond the last boundary
    cen, bnd = _tables(nbits)
    packed = torch.full((n // 32 * nbits,), -1, dtype=torch.int32, device=DEV)
    result = torch.zeros(4, device=DEV)
    work = torch.zeros(capi.eden_work_doubles(n), dtype=torch.float64, device=DEV)
    capi.eden_quantize(x.to(DEV), bnd, cen, nbits, packed, result, work)
    bins_o, res_o = oracle.eden_quantize(x.numpy(), GOLD["boundaries_%d" % nbits], GOLD["centroids_%d" % nbits], nbits)
    assert (result.cpu().numpy().view(np.uint32) == res_o.view(np.uint32)).all()
    assert (packed.cpu().numpy().view(np.uint32) == oracle.bins_to_bits(bins_o, nbits)).all()
    out = torch.zeros(n, device=DEV)
    capi.eden_dequantize(packed, n, cen, nbits, out)
    assert (out.cpu().numpy() == oracle.eden_dequantize(bins_o, GOLD["centroids_%d" % nbits])).all()


def test_eden_quantize_degenerate_norms(capi, oracle):
    """all zeros (0/0 -> NaN: torch.bucketize's lower bound sends it to the last bin) and a norm outside the fast-division range"""
    cen, bnd = _tables(4)
    for x in (torch.zeros(64), torch.full((64,), 1e-30), torch.full((64,), 3e18) * torch.randn(64).sign()):
        packed = torch.zeros(8, dtype=torch.int32, device=DEV)
        result = torch.zeros(4, device=DEV)
        work = torch.zeros(capi.eden_work_doubles(64), dtype=torch.float64, device=DEV)
        capi.eden_quantize(x.to(DEV), bnd, cen, 4, packed, result, work)
        bins_o, res_o = oracle.eden_quantize(x.numpy(), GOLD["boundaries_4"], GOLD["centroids_4"], 4)
        got, want = result.cpu().numpy(), res_o
        same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
        assert same.all()
        assert (packed.cpu().numpy().view(np.uint32) == oracle.bins_to_bits(bins_o, 4)).all()


@pytest.mark.parametrize("case", [tuple(c) for c in GOLD["cases"]])
def test_eden_class_against_reference_outputs(capi, oracle, case):
    """Eden.compress / decompress with the reference's tables vs what the reference produced on the CPU"""
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    dim, nbits, seed, nslices = (int(v) for v in case)
    cen = {nbits: torch.from_numpy(GOLD["centroids_%d" % nbits])}
    bnd = {nbits: torch.from_numpy(GOLD["boundaries_%d" % nbits])}
    eden = Eden(centroids=cen, boundaries=bnd, device=DEV)
    x = torch.from_numpy(GOLD["x_%d" % dim])
    data = eden.compress(x.to(DEV), nbits, seed)
    assert len(data) == nslices
    key = "%d_%d_%d" % (dim, nbits, seed)
    for k, d in enumerate(data):
        scale_g, orig_g, nh_g = GOLD["meta_%s_%d" % (key, k)]
        assert (d["orig_dim"], d["num_hadamard"], d["nbits"], d["seed"]) == (int(orig_g), int(nh_g), nbits, seed)
        bins = oracle.bits_to_bins(d["packed_bins"].cpu().numpy().view(np.uint32), nbits)
        bins_g = oracle.bits_to_bins(GOLD["packed_%s_%d" % (key, k)].view(np.uint32), nbits)
        assert (bins != bins_g).mean() <= 2e-3 and (np.abs(bins - bins_g) <= 1).all()
        assert abs(float(d["scale"]) - scale_g) <= 1e-4 * abs(scale_g)
    rec = eden.decompress(data).cpu()
    rec_g = torch.from_numpy(GOLD["rec_" + key])
    assert rec.shape == rec_g.shape and rec.dtype == x.dtype
    nmse = float(((rec - x) ** 2).sum() / (x ** 2).sum())
    nmse_g = float(((rec_g - x) ** 2).sum() / (x ** 2).sum())
    assert abs(nmse - nmse_g) <= 5e-3 * nmse_g
    assert float(((rec - rec_g) ** 2).sum() / (x ** 2).sum()) <= 2e-2 * nmse_g + 1e-9


def test_eden_class_own_tables_and_large_vector():
    """the computed Lloyd-Max tables give the textbook distortion D (with EDEN's unbiased scale ||x||^2 / <c, x> the
    NMSE is D / (1 - D)); a 2^22 vector goes through the multi-pass transform"""
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    eden = Eden(device=DEV)
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.randn(1 << 22, generator=g, device=DEV) * 1e-3
    from dynamiq_sigcomm_artifact_amd.eden import lloyd_max_normal, _conditional_means
    textbook = {1: 0.3634, 2: 0.1175, 4: 0.009497}     # Lloyd-Max distortion of N(0,1): Max (1960), tables I-II
    for nbits in (1, 2, 4, 8):
        c = lloyd_max_normal(nbits)
        # at the stationary point E[c(X) X] = E[c(X)^2], so D = 1 - E[c^2]; cell masses from the cdf
        from scipy.stats import norm
        b = np.concatenate(([-np.inf], (c[:-1] + c[1:]) / 2, [np.inf]))
        d = 1.0 - float(np.sum(c * c * (norm.cdf(b[1:]) - norm.cdf(b[:-1]))))
        if nbits in textbook:
            assert abs(d - textbook[nbits]) < 5e-5
        rec = eden.decompress(eden.compress(x, nbits, 7))
        nmse = float(((rec - x) ** 2).sum() / (x ** 2).sum())
        assert abs(nmse - d / (1 - d)) <= 0.02 * d, (nbits, nmse, d)
    odd = torch.randn(3000, generator=g, device=DEV).to(torch.bfloat16)
    rec = eden.decompress(eden.compress(odd, 4, 1))
    assert rec.dtype == torch.bfloat16 and rec.numel() == 3000
    assert float(((rec.float() - odd.float()) ** 2).sum() / (odd.float() ** 2).sum()) < 0.02


def _thc_torch_chain(rotated, lo, delta, levels, uniform):
    """thc_hooks.py:161-166 with bernoulli_(p) spelled (uniform < p)"""
    r = rotated.clone()
    r.sub_(lo).div_(delta)
    r.clamp_(min=0, max=levels - 1)
    floored = r.floor()
    probs = r.sub_(floored)
    floored.add_((uniform < probs).float())
    return floored.to(torch.bfloat16)


def test_thc_kernels_bit_exact(capi, oracle):
    n = 100003
    g = torch.Generator().manual_seed(2)
    rot = torch.randn(n, generator=g) * 0.01
    rot[3] = float("inf")
    rot[4] = float("-inf")
    rot[5] = float("nan")
    rot[6] = 0.0
    uni = torch.rand(n, generator=g)
    uni[::13] = 0.0
    max_norm = torch.tensor(0.3)
    lo = (-(3.2971933456919635 * max_norm / math.sqrt(1024))).reshape(1)
    for levels in (16, 31, 64):
        delta = ((-lo - lo) / (levels - 1) + 1e-23).reshape(1)
        out = torch.zeros(n, dtype=torch.bfloat16, device=DEV)
        capi.thc_quantize(rot.to(DEV), uni.to(DEV), out, lo.to(DEV), delta.to(DEV), levels)
        want = oracle.thc_quantize(rot.numpy(), uni.numpy(), float(lo), float(delta), levels)
        got = to_bits(out)
        nan = (got & 0x7fff) > 0x7f80
        assert ((got == want) | (nan & ((want & 0x7fff) > 0x7f80))).all()
        chain = _thc_torch_chain(rot.to(DEV), lo.to(DEV), delta.to(DEV), levels, uni.to(DEV))
        keep = ~torch.isnan(chain.float())
        assert torch.equal(out[keep], chain[keep])
        # decode: (sum of levels) * (delta / W) + lo
        step = (delta / 4).reshape(1)
        dec = torch.zeros(n, device=DEV)
        capi.thc_dequantize(out, dec, step.to(DEV), lo.to(DEV))
        want_d = oracle.thc_dequantize(want, float(step), float(lo))
        ok = (dec.cpu().numpy().view(np.uint32) == want_d.view(np.uint32)) | np.isnan(want_d)
        assert ok.all()
        ref = out.float().mul_(step.to(DEV)).add_(lo.to(DEV))
        assert torch.equal(dec[keep], ref[keep])


def test_thc_compressor_round_trip():
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    size = 100000
    d = 1 << 17
    params = {"d": {(0, 0): d}, "size": {(0, 0): size}, "T": 3.2971933456919635, "nclients": 1, "rank": 0,
              "quantization_levels": 64, "device": DEV}
    comp = OldINCACudaHadamardCompressor(params)
    g = torch.Generator(device=DEV).manual_seed(1)
    x = (torch.randn(size, generator=g, device=DEV) * 1e-3).to(torch.bfloat16)
    norm = x.float().norm(2)
    levels = comp.compress(x, (0, 0), norm)
    assert levels.dtype == torch.bfloat16 and levels.numel() == d
    assert float(levels.float().min()) >= 0 and float(levels.float().max()) <= 63
    assert torch.equal(levels.float(), levels.float().round())
    rec = comp.decompress(levels, (0, 0), norm)
    assert rec.numel() == size
    nmse = float(((rec - x.float()) ** 2).sum() / (x.float() ** 2).sum())
    # per rotated coordinate (unit variance after scaling by sqrt(d)/||x||): uniform stochastic rounding with step
    # 2T/63 adds step^2/6, clipping at +-T adds E[(|z|-T)^2; |z|>T] = 2((1+T^2) Q(T) - T phi(T)); only size of the d
    # inverse-rotated coordinates are kept
    from scipy.stats import norm as gauss
    T = 3.2971933456919635
    expect = ((2 * T / 63) ** 2 / 6 + 2 * ((1 + T * T) * gauss.sf(T) - T * gauss.pdf(T))) * size / d
    assert abs(nmse - expect) < 0.03 * expect
    # the sum over two ranks decodes with delta / 2
    params2 = dict(params, nclients=2)
    c0, c1 = OldINCACudaHadamardCompressor(dict(params2, rank=0)), OldINCACudaHadamardCompressor(dict(params2, rank=1))
    y = (torch.randn(size, generator=g, device=DEV) * 1e-3).to(torch.bfloat16)
    big = torch.maximum(norm, y.float().norm(2))
    total = (c0.compress(x, (0, 0), big).float() + c1.compress(y, (0, 0), big).float()).to(torch.bfloat16)
    mean = c0.decompress(total, (0, 0), big)
    ref = (x.float() + y.float()) / 2
    assert float(((mean - ref) ** 2).sum() / (ref ** 2).sum()) < 0.02


def test_binding_functions(eden_utils, capi):
    n, nbits = 4096, 4
    cen, bnd = _tables(nbits)
    x = torch.randn(n, device=DEV) * 1e-3
    packed, result = eden_utils.eden_quantize(x, bnd, cen, nbits)
    packed2 = torch.empty_like(packed)
    result2 = torch.empty_like(result)
    capi.eden_quantize(x, bnd, cen, nbits, packed2, result2, torch.empty(capi.eden_work_doubles(n), dtype=torch.float64, device=DEV))
    assert torch.equal(packed, packed2) and torch.equal(result, result2)
    out = eden_utils.eden_dequantize(packed, cen, nbits)
    assert out.shape == (n,) and bool(torch.isin(out, cen).all())
    lo, delta = torch.tensor([-0.005], device=DEV), torch.tensor([0.01 / 63], device=DEV)
    u = torch.rand(n, device=DEV)
    lev = eden_utils.thc_quantize(x, u, lo, delta, 64)
    lev2 = torch.empty_like(lev)
    capi.thc_quantize(x, u, lev2, lo, delta, 64)
    assert torch.equal(lev, lev2)
    dec = torch.empty(n, device=DEV)
    eden_utils.thc_dequantize(lev, dec, delta, lo)
    assert float((dec - x).abs().max()) <= float(delta) * 1.01
    with pytest.raises(RuntimeError, match="vec size must be a positive multiple of 32"):
        eden_utils.eden_quantize(x[:100].contiguous(), bnd, cen, nbits)
    with pytest.raises(RuntimeError, match="boundaries must hold"):
        eden_utils.eden_quantize(x, bnd[:5].contiguous(), cen, nbits)


@pytest.mark.parametrize("levels", [2, 64, 256])
@pytest.mark.parametrize("n", [1 << 16, 1 << 20])
def test_thc_levels_where_the_comparison_is_a_tie(capi, n, levels):
    """uniform values equal to the fraction they are compared with, their neighbours, 0 and 1, and rotated values on, next to and
    beyond the grid's ends: the levels of the folded quantiser are those of the quantiser that divides"""
    g = torch.Generator().manual_seed(n + levels)
    x = (torch.randn(n, generator=g) * 1e-2).to(DEV)
    x[7] = 3.0                                                              # (a spike moves whole columns beyond the ends)
    scale = float(np.float32(1.0) / np.float32(np.sqrt(n)))
    rot = x.clone()
    capi.rht_blocked(rot, None, n, scale, False)
    hi = 1.5 * float(rot.std())
    lo = torch.tensor([-hi], dtype=torch.float32, device=DEV)
    delta = torch.tensor([2 * hi / (levels - 1)], dtype=torch.float32, device=DEV)
    q = ((rot - lo) / delta).clamp(0, levels - 1)
    frac = q - q.floor()
    k = torch.arange(n, device=DEV) % 6
    uni = torch.where(k == 0, frac, torch.where(k == 1, torch.nextafter(frac, torch.ones_like(frac)), torch.where(
        k == 2, torch.nextafter(frac, -torch.ones_like(frac)).clamp(min=0), torch.where(k == 3, torch.zeros_like(frac), torch.where(
            k == 4, torch.full_like(frac, 1 - 2.0 ** -24), 1 - frac)))))
    for bad in (None, float("nan"), float("inf")):
        if bad is not None:
            rot.fill_(bad)
            x[0] = bad
        want, got = torch.empty(n, dtype=torch.bfloat16, device=DEV), torch.empty(n, dtype=torch.bfloat16, device=DEV)
        work = x.clone()
        if bad is not None:
            rot = x.clone()
            capi.rht_blocked(rot, None, n, scale, False)
        capi.thc_quantize(rot, uni, want, lo, delta, levels)
        capi.thc_rht_quantize(work, None, uni, got, n, scale, lo, delta, levels)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), bad


@pytest.mark.parametrize("n", [1 << 16, 1 << 20])
@pytest.mark.parametrize("delta", [2.0 ** -149, 2.0 ** -126, 2.0 ** 126, 2.0 ** 126 * 1.25, 2.0 ** 127 * 1.9])
def test_thc_levels_of_the_widest_and_the_finest_grid(capi, n, delta):
    """a spacing whose reciprocal is no ordinary float32: the levels of the folded quantiser are those of the quantiser that
    divides"""
    levels = 64 if delta < 1.0 else 4
    g = torch.Generator().manual_seed(n)
    x = (torch.randn(n, generator=g) * (delta * 0.15 / math.sqrt(n))).to(DEV)
    if delta < 1.0:
        x = (torch.randint(-1, 2, (n,), generator=g).float() * 2.0 ** -149).to(DEV)
    rot = x.clone()
    capi.rht_blocked(rot, None, n, 1.0, False)
    lo = torch.tensor([-delta if delta > 1.0 else -32 * delta], dtype=torch.float32, device=DEV)
    step = torch.tensor([delta], dtype=torch.float32, device=DEV)
    q = ((rot.double() - lo.double()) / delta).clamp(0, levels - 1)
    frac = (q - q.floor()).float()
    uni = torch.where(torch.arange(n, device=DEV) % 2 == 0, frac, torch.rand(n, generator=g).to(DEV))
    want, got = torch.empty(n, dtype=torch.bfloat16, device=DEV), torch.empty(n, dtype=torch.bfloat16, device=DEV)
    capi.thc_quantize(rot, uni, want, lo, step, levels)
    capi.thc_rht_quantize(x, None, uni, got, n, 1.0, lo, step, levels)
    assert torch.isfinite(rot).float().mean() > 0.9 and want.unique().numel() > 2
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dim", [1 << k for k in range(18, 27)])
def test_thc_draws_what_torch_would_draw(dim):
    """compress without uniform values: the levels are those of values that uniform_ drew from a generator in the same state, call
    after call, and the generator ends where uniform_ leaves it; lengths on either side of those that the kernel draws for"""
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    key, used = (0, 0), dim - 77
    params = {"d": {key: dim}, "size": {key: used}, "seed": 42, "T": 3.0, "device": DEV, "quantization_levels": 64, "nclients": 4, "rank": 1}
    a, b = OldINCACudaHadamardCompressor(params), OldINCACudaHadamardCompressor(params)
    for codec in (a, b):                                        # (a seed and an offset with high words)
        codec.sender_prng.manual_seed(0x1234567890ABCDEF)
        codec.sender_prng.set_offset((1 << 34) - 4)
    x = torch.randn(used, generator=torch.Generator(device=DEV).manual_seed(dim), device=DEV)
    norm = x.norm()
    for _ in range(3):
        got = a.compress(x, key, norm)
        uni = torch.empty(dim, device=DEV).uniform_(0.0, 1.0, generator=b.sender_prng)
        want = b.compress(x, key, norm, uniform=uni)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        assert a.sender_prng.get_offset() == b.sender_prng.get_offset()
        assert torch.equal(a.sender_prng.get_state(), b.sender_prng.get_state())


@pytest.mark.parametrize("dim,row", [(1 << 19, 1 << 11), (1 << 22, 1 << 14), (1 << 23, 1 << 13), (1 << 25, 1 << 15)])
def test_thc_draws_behind_a_short_source(dim, row):
    """sources that end at, before and behind a row of the strided pass, a wave's rows and a thread's: the rows behind them are neither
    written nor read where the values are drawn, whatever lies there, and the levels are those of the pass that reads them all"""
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    key = (0, 0)
    x = torch.randn(dim, generator=torch.Generator(device=DEV).manual_seed(dim), device=DEV)
    for used in (1, row, row + 1, 16 * row, 32 * row - 3, 33 * row + 5, 64 * row, dim // 2 + 1, dim - row - 1, dim - row, dim - 1):
        params = {"d": {key: dim}, "size": {key: used}, "seed": 42, "T": 3.0, "device": DEV, "quantization_levels": 64, "nclients": 4, "rank": 1}
        a, b = OldINCACudaHadamardCompressor(params), OldINCACudaHadamardCompressor(params)
        a._buffer(key, "work").fill_(float("nan"))
        norm = x[:used].norm()
        got = a.compress(x[:used], key, norm)
        want = b.compress(x[:used], key, norm, uniform=torch.empty(dim, device=DEV).uniform_(0.0, 1.0, generator=b.sender_prng))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), used


def test_thc_recorded_draws_are_torchs():
    """a graph that holds a compress call draws through the generator's registered state: every replay other values, those of an
    eager call from the same state"""
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    key, dim = (0, 0), 1 << 20
    params = {"d": {key: dim}, "size": {key: dim}, "seed": 42, "T": 3.0, "device": DEV, "quantization_levels": 64, "nclients": 4, "rank": 0}
    a, b = OldINCACudaHadamardCompressor(params), OldINCACudaHadamardCompressor(params)
    x = torch.randn(dim, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    norm = x.norm()
    a.compress(x, key, norm)
    b.compress(x, key, norm)
    graph = torch.cuda.CUDAGraph()
    graph.register_generator_state(a.sender_prng)
    with torch.cuda.graph(graph):
        got = a.compress(x, key, norm)
    for _ in range(3):
        graph.replay()
        want = b.compress(x, key, norm)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("blocks", [1, 3, 32])
def test_few_blocks_of_2p15_are_those_of_a_long_vector(capi, blocks):
    """up to 32 blocks of 2^15 take two passes, more of them one: the same bits, with packed and float signs, either way, and with THC's
    quantisers at the ends"""
    block, levels = 1 << 15, 64
    n, many = blocks * block, 40 * block
    g = torch.Generator(device=DEV).manual_seed(blocks)
    x = torch.randn(many, generator=g, device=DEV)
    sign = torch.randint(0, 2, (many,), generator=g, device=DEV).float() * 2.0 - 1.0
    scale = 1.0 / block ** 0.5
    for packed in (False, True):
        for inverse in (False, True):
            long, few = x.clone(), x[:n].clone()
            capi.rht_blocked(long, capi.pack_signs(sign) if packed else sign, block, scale, inverse)
            capi.rht_blocked(few, capi.pack_signs(sign[:n]) if packed else sign[:n], block, scale, inverse)
            assert torch.equal(few.view(torch.int32), long[:n].view(torch.int32)), (packed, inverse)
    odd = torch.zeros(n + 1, device=DEV)[1:].copy_(x[:n])       # off the 16 bytes: two passes as well
    capi.rht_blocked(odd, sign[:n], block, scale, True)
    long = x.clone()
    capi.rht_blocked(long, sign, block, scale, True)
    assert torch.equal(odd.view(torch.int32), long[:n].view(torch.int32))
    lo, step = torch.tensor([-3.0], device=DEV), torch.tensor([6.0 / (levels - 1)], device=DEV)
    uni, bits = torch.rand(n, generator=g, device=DEV), capi.pack_signs(sign[:n])
    long, few = x.clone(), x[:n].clone()
    capi.rht_blocked(long, sign, block, scale, False)
    want, got = (torch.empty(n, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    capi.thc_quantize(long[:n].contiguous(), uni, want, lo, step, levels)
    capi.thc_rht_quantize(few, bits, uni, got, block, scale, lo, step, levels)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and want.unique().numel() > 32
    back = torch.zeros(many, device=DEV)
    out = torch.empty(n, device=DEV)
    capi.thc_dequantize(want, out, step, lo)
    back[:n] = out
    capi.rht_blocked(back, sign, block, scale, True)
    capi.thc_dequantize_irht(want, bits, out, block, scale, step, lo)
    assert torch.equal(out.view(torch.int32), back[:n].view(torch.int32))


@pytest.mark.parametrize("bits,shift", [(14, 0), (16, 1), (17, 0), (18, 3), (21, 0), (24, 1), (26, 0), (27, 0), (30, 0)])
def test_long_transforms_of_a_unit_vector(capi, bits, shift):
    """H e_k = (-1)^popcount(j & k): every element of the contiguous pass and of strided passes of four to ten row bits, on vectors
    that start anywhere"""
    n = 1 << bits
    k = 0x2D5B3A97 & (n - 1)
    x = torch.zeros(n + shift, device=DEV)[shift:]
    x[k] = 0.5
    capi.rht_blocked(x, None, n, 2.0, False)
    piece = 1 << min(bits, 26)
    for at in range(0, n, piece):
        j = torch.arange(at, at + piece, dtype=torch.int32, device=DEV) & k
        for s in (16, 8, 4, 2, 1):
            j ^= j >> s
        assert torch.equal(x[at:at + piece], 1.0 - 2.0 * (j & 1).float()), at


@pytest.mark.parametrize("n,block", [(64, 64), (1024, 1024), (1024, 64), (1 << 15, 1 << 15), (1 << 16, 1 << 16),
                                     (1 << 17, 1 << 17), (1 << 20, 1 << 20), (1 << 22, 1 << 22), (1 << 23, 1 << 23), (1 << 18, 1 << 12), (3 << 14, 1 << 14)])
def test_thc_quantiser_folded_into_the_transform(capi, n, block):
    """dq_thc_rht_quantize == rht_blocked + thc_quantize and dq_thc_dequantize_irht == thc_dequantize + inverse
    rht_blocked, bit for bit, for single-pass and multi-pass transforms"""
    g = torch.Generator().manual_seed(n + block)
    x = (torch.randn(n, generator=g) * 1e-2).to(DEV)
    sign = (torch.randint(0, 2, (n,), generator=g).float() * 2 - 1).to(DEV)
    uni = torch.rand(n, generator=g).to(DEV)
    scale = float(np.float32(1.0) / np.float32(np.sqrt(block)))
    norm = float(x.norm())
    T, levels = 2.5, 31
    hi = T * norm / np.sqrt(n)
    lo = torch.tensor([-hi], dtype=torch.float32, device=DEV)
    delta = torch.tensor([2 * hi / (levels - 1) + 1e-23], dtype=torch.float32, device=DEV)
    rot = x.clone()
    capi.rht_blocked(rot, sign, block, scale, False)
    want = torch.empty(n, dtype=torch.bfloat16, device=DEV)
    capi.thc_quantize(rot, uni, want, lo, delta, levels)
    work = x.clone()
    got = torch.empty(n, dtype=torch.bfloat16, device=DEV)
    capi.thc_rht_quantize(work, sign, uni, got, block, scale, lo, delta, levels)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert int(want.float().max()) <= levels - 1 and float(want.float().std()) > 1.0       # the quantiser did something
    # the way back, as after a direct sum over 4 ranks
    summed = (want.float() * 4).to(torch.bfloat16)
    step = delta / 4
    dec = torch.empty(n, device=DEV)
    capi.thc_dequantize(summed, dec, step, lo)
    capi.rht_blocked(dec, sign, block, scale, True)
    back = torch.full((n,), 7.0, device=DEV)
    capi.thc_dequantize_irht(summed, sign, back, block, scale, step, lo)
    assert torch.equal(back.view(torch.int32), dec.view(torch.int32))
    # the diagonal as packed bits: the same levels, the same vector back, the same rotation
    bits = capi.pack_signs(sign)
    work.copy_(x)
    got.zero_()
    capi.thc_rht_quantize(work, bits, uni, got, block, scale, lo, delta, levels)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    back.fill_(7.0)
    capi.thc_dequantize_irht(summed, bits, back, block, scale, step, lo)
    assert torch.equal(back.view(torch.int32), dec.view(torch.int32))
    rot2 = x.clone()
    capi.rht_blocked(rot2, bits, block, scale, False)
    assert torch.equal(rot2.view(torch.int32), rot.view(torch.int32))
    capi.rht_blocked(rot2, bits, block, scale, True)
    capi.rht_blocked(rot, sign, block, scale, True)
    assert torch.equal(rot2.view(torch.int32), rot.view(torch.int32))
    # buffers that are only element-aligned take the scalar paths
    if n <= 1 << 16:
        r3 = torch.zeros(n + 4, device=DEV)[1:1 + n].copy_(x)
        r4 = r3.clone()
        capi.rht_blocked(r3, bits, block, scale, False)
        capi.rht_blocked(r4, sign, block, scale, False)
        assert torch.equal(r3.view(torch.int32), r4.view(torch.int32))
        w2 = torch.zeros(n + 4, device=DEV)[1:1 + n].copy_(x)
        u2 = torch.zeros(n + 4, device=DEV)[3:3 + n].copy_(uni)
        g2 = torch.zeros(n + 4, dtype=torch.bfloat16, device=DEV)[1:1 + n]
        capi.thc_rht_quantize(w2, sign, u2, g2, block, scale, lo, delta, levels)
        assert torch.equal(g2.view(torch.int16), want.view(torch.int16))
        b2 = torch.zeros(n + 4, device=DEV)[1:1 + n]
        capi.thc_dequantize_irht(g2 * 4, sign, b2, block, scale, step, lo)
        assert torch.equal(b2.view(torch.int32), dec.view(torch.int32))


@pytest.mark.parametrize("nbits", [1, 3, 4, 8])
@pytest.mark.parametrize("n,block", [(32, 32), (96, 32), (1024, 1024), (4096 * 3, 4096), (1 << 15, 1 << 15), (1 << 16, 1 << 16),
                                     (1 << 17, 1 << 17), (1 << 20, 1 << 20), (1 << 22, 1 << 22), (1 << 23, 1 << 23), (1 << 18, 1 << 12)])
def test_eden_dequantiser_folded_into_the_inverse_transform(capi, nbits, n, block):
    """dq_eden_dequantize_irht == eden_dequantize, inverse rht_blocked, product with the scale -- bit for bit, single-pass
    and multi-pass transforms, float and packed diagonals, with and without the scale"""
    g = torch.Generator().manual_seed(n + nbits)
    cen, _ = _tables(nbits)
    bins = torch.randint(0, 1 << nbits, (n,), generator=g, dtype=torch.int32).to(DEV)
    packed = torch.empty(n // 32 * nbits, dtype=torch.int32, device=DEV)
    capi.bins_to_bits(bins, packed, nbits)
    sign = (torch.randint(0, 2, (n,), generator=g).float() * 2 - 1).to(DEV)
    scale = float(np.float32(1.0) / np.float32(np.sqrt(block)))
    eden_scale = torch.tensor([0.00123], dtype=torch.float32, device=DEV)
    want = torch.empty(n, device=DEV)
    capi.eden_dequantize(packed, n, cen, nbits, want)
    capi.rht_blocked(want, sign, block, scale, True)
    for sg in (sign, capi.pack_signs(sign), None):
        ref = want
        if sg is None:
            ref = torch.empty(n, device=DEV)
            capi.eden_dequantize(packed, n, cen, nbits, ref)
            capi.rht_blocked(ref, None, block, scale, True)
        got = torch.full((n + 8,), 7.0, device=DEV)
        capi.eden_dequantize_irht(packed, n, cen, nbits, sg, got[:n], block, scale)
        assert torch.equal(got[:n].view(torch.int32), ref.view(torch.int32)) and bool((got[n:] == 7.0).all())
        capi.eden_dequantize_irht(packed, n, cen, nbits, sg, got[:n], block, scale, post_scale=eden_scale)
        assert torch.equal(got[:n].view(torch.int32), (eden_scale * ref).view(torch.int32)) and bool((got[n:] == 7.0).all())


def test_srrcomp_utils_surface(capi, oracle):
    """the helpers srrcomp.Eden inherits from SRRCompUtils (srrcomp.py:13-167) and its _quantize (:356-361), as methods
    of the drop-in class: each equals the oracle's function or the entry point it wraps"""
    from dynamiq_sigcomm_artifact_amd.eden import Eden, SRRCompUtils
    eden = Eden(device=DEV)
    assert isinstance(eden, SRRCompUtils) and set(eden.utils) == {"cpu", "gpu"}
    assert set(eden.utils["gpu"]) == {"Hadamard", "BinsToBits", "BitsToBins"}
    with pytest.raises(Exception, match="Illegal gpuacctype"):
        SRRCompUtils("opencl")
    with pytest.raises(RuntimeError, match="device tensors only"):
        eden.utils["cpu"]["Hadamard"](torch.zeros(8))
    # randDiag: the integer hash of the reference; with torchRNG torch's own stream of +-1
    for size, seed in ((1000, 7), (4096, 123456789), (1, 0)):
        got = eden.randDiag(size, DEV, seed)
        assert got.dtype == torch.float32 and np.array_equal(got.cpu().numpy(), oracle.rand_diag(size, seed))
    coins = eden.randDiag(512, DEV, 5, torchRNG=True)
    assert set(coins.cpu().tolist()) == {-1.0, 1.0} and torch.equal(coins, eden.randDiag(512, DEV, 5, torchRNG=True))
    # Hadamard: in place, returns the flat view
    x = torch.randn(1 << 12, generator=torch.Generator().manual_seed(3))
    x_d = x.to(DEV).view(64, 64)
    y = eden.Hadamard(x_d)
    assert y.data_ptr() == x_d.data_ptr() and np.array_equal(y.cpu().numpy(), oracle.fwht(x.numpy()))
    with pytest.raises(Exception, match="power of 2"):
        eden.Hadamard(torch.zeros(12, device=DEV))
    # the packers take the int64 bins of torch.bucketize
    bins = torch.randint(0, 32, (4096,), generator=torch.Generator().manual_seed(4))
    bits = eden.EdenBinsToBits(bins.to(DEV), 5)
    assert bits.dtype == torch.int32 and np.array_equal(bits.cpu().numpy().view(np.uint32), oracle.bins_to_bits(bins.numpy().astype(np.int32), 5).view(np.uint32))
    assert torch.equal(eden.EdenBitsToBins(bits, 5).cpu(), bins.to(torch.int32))
    # _quantize: the bins and the scale of eden_quantize
    n, nbits = 8192, 4
    v = torch.randn(n, generator=torch.Generator().manual_seed(6)).to(DEV)
    q_bins, scale = eden._quantize(v, nbits)
    cen, bnd = eden._tables(nbits)
    packed = torch.empty(n // 32 * nbits, dtype=torch.int32, device=DEV)
    result = torch.empty(4, dtype=torch.float32, device=DEV)
    capi.eden_quantize(v, bnd, cen, nbits, packed, result, torch.empty(capi.eden_work_doubles(n), dtype=torch.float64, device=DEV))
    assert q_bins.dtype == torch.int64 and torch.equal(eden.EdenBinsToBits(q_bins, nbits), packed)
    assert float(scale) == float(result[2])
    # against torch's own ops away from the boundaries: at most a handful of bins differ by the rounding of the quotient
    ref = torch.bucketize(v * (n ** 0.5) / torch.norm(v, 2), bnd)
    assert int((ref != q_bins).sum()) <= 2


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 33, 1000, 1024, 1500, 4097, 32768 - 7, 65536, 100003, (1 << 22) + (1 << 20), (1 << 23) - 5])
def test_slices_in_one_call_equal_the_single_calls(capi, n, dt):
    """compress and decompress of a vector whose slices are tiny, ragged, of one pass and of two, with drawn and with written
    diagonals, aligned and not, against the calls they stand for: padding, rand_diag, rht_blocked, eden_quantize; and back"""
    import math
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    dev = "cuda:0"
    eden = Eden(device=dev)
    g = torch.Generator(device=dev).manual_seed(n)
    nbits, seed = 3 + n % 3, 17
    vec = (torch.randn(n + 1, generator=g, device=dev) * 1e-2).to(dt)[n & 1:][:n]
    print("case", n, dt, flush=True)
    data = eden.compress(vec, nbits, seed)
    assert sum(d["orig_dim"] for d in data) == n
    centroids, boundaries = eden._tables(nbits)
    at, want = 0, []
    for d in data:
        size = d["packed_bins"].numel() // nbits * 32
        inv = float(np.float32(1.0) / np.float32(math.sqrt(size)))
        x = torch.zeros(size, device=dev)
        x[:d["orig_dim"]] = vec[at:at + d["orig_dim"]].float()
        at += d["orig_dim"]
        diags = []
        for i in range(d["num_hadamard"]):
            diags.append(torch.empty(size, device=dev))
            capi.rand_diag(diags[-1], seed + i)
            capi.rht_blocked(x, diags[-1], size, inv, False)
        packed = torch.empty(size // 32 * nbits, dtype=torch.int32, device=dev)
        result = torch.empty(4, device=dev)
        capi.eden_quantize(x, boundaries, centroids, nbits, packed, result, torch.empty(capi.eden_work_doubles(size), dtype=torch.float64, device=dev))
        assert torch.equal(packed, d["packed_bins"]) and torch.equal(result[2].view(torch.int32), d["scale"].view(torch.int32))
        y = torch.empty(size, device=dev)
        capi.eden_dequantize(packed, size, centroids, nbits, y)
        for diag in reversed(diags):
            capi.rht_blocked(y, diag, size, inv, True)
        want.append((result[2] * y)[:d["orig_dim"]].to(dt))
    got = eden.decompress(data)
    assert got.dtype == dt and torch.equal(got, torch.cat(want))


@pytest.mark.parametrize("sizes", [(1 << 14, 1 << 15), (1 << 14, 1 << 18, 1 << 22), (1 << 17,), (1 << 19, 1 << 14), (1 << 21, 1 << 20),
                                   (1 << 23,), (1 << 24,), (1 << 25,), (1 << 26,)])
def test_scale_from_the_sums_of_the_last_pass(sizes):
    """EDEN's scale is (norm * norm) / dot of float32s, and the sum of squares behind the norm comes out of the last pass of the
    rotation: for every number of rows of that pass (16 ones beside longer slices, up to 1024, and 64 behind another strided
    pass) against the exact sums of the rotated values.  Three roundings to float32 of sums in double: 2^-22."""
    import math
    from dynamiq_sigcomm_artifact_amd import capi
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    dev, nbits, seed = "cuda:0", 4, 5
    eden = Eden(device=dev)
    vec = torch.randn(sum(sizes), generator=torch.Generator(device=dev).manual_seed(1), device=dev) * 1e-2
    centroids, boundaries = eden._tables(nbits)
    slices, at = [], 0
    for n in sizes:
        slices.append((at, n, n, 1))
        at += n
    parts = capi.host().eden_compress(vec, boundaries, centroids, nbits, seed, slices)
    for (packed, scale), (at, n, _, _) in zip(parts, slices):
        x = vec[at:at + n].clone()
        diag = torch.empty(n, device=dev)
        capi.rand_diag(diag, seed)
        capi.rht_blocked(x, diag, n, float(np.float32(1.0) / np.float32(math.sqrt(n))), False)
        bins = eden.EdenBitsToBins(packed, nbits).to(torch.int64)
        exact = x.double()
        want = (exact * exact).sum() / (centroids[bins].double() * exact).sum()
        assert abs(float(scale) / float(want) - 1.0) < 2.0 ** -22, (n, float(scale), float(want))


def _sum_on_a_boundary(bits, shift, which, k):
    """A vector of 2^bits elements, an even number of bits, whose rotation by H / sqrt(n) is 1,024 values, each in as many places,
    with a sum of squares within 2^-53 of the middle between two float32s: to which of them it rounds depends on the order in which
    a double adds the squares.  The 1,024 values are u + b and u - b: u, 512 of them, are whole numbers and exact, b has more
    fractional digits than a sum of the two keeps (found by trying 2^33 pairs of u and b).  They stay the same with the digits of
    their index in another order and with the signs of any character of it, and lie `shift` digits up in the vector's index."""
    seed, b = ((687, 14603885), (1143, 13973873), (1523, 13967869), (2132, 14500689))[which]
    x = np.zeros(1024, np.float32)
    x[:512] = np.random.default_rng(seed).integers(-2048, 2049, 512)
    x[512] = b * 2.0 ** -9
    rng = np.random.default_rng([bits, shift, which, k])
    order, character = rng.permutation(9), int(rng.integers(1024))
    i = np.arange(1024)
    source, sign = i & 512, np.ones(1024, np.float32)
    for new, old in enumerate(order):
        source |= ((i >> new) & 1) << old
    for d in range(10):
        if character >> d & 1:
            sign[(i >> d) & 1 == 1] *= -1.0
    out = np.zeros(1 << bits, np.float32)
    out[i << shift] = x[source] * sign
    return out


@pytest.mark.parametrize("bits", [14, 16, 18, 20, 22, 24, 26])
def test_scale_is_the_slices_own(capi, oracle, bits):
    """the sums behind a slice's scale, and so its bins, are the same alone, beside longer and shorter slices, in eden_quantize
    and in the oracle, also where the order of the additions decides the last bit"""
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    n, nbits, seed = 1 << bits, 4, 5
    eden = Eden(device=DEV)
    centroids, boundaries = eden._tables(nbits)
    diag = torch.empty(n, device=DEV)
    capi.rand_diag(diag, seed)
    others = torch.randn(1 << 22, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    for shift in sorted({0, (bits - 10) // 2, bits - 10}):
        for k in range(16 if bits <= 18 else 4 if bits <= 22 else 2):
            x = torch.from_numpy(_sum_on_a_boundary(bits, shift, k % 4, k)).to(DEV) * diag
            y = x.clone()
            capi.rht_blocked(y, diag, n, 2.0 ** (-bits // 2), False)
            packed = torch.empty(n // 32 * nbits, dtype=torch.int32, device=DEV)
            result = torch.empty(4, device=DEV)
            work = torch.empty(capi.eden_work_doubles(n), dtype=torch.float64, device=DEV)
            capi.eden_quantize(y, boundaries, centroids, nbits, packed, result, work)
            if bits <= 24 or k == 0:
                bins_o, res_o = oracle.eden_quantize(y.cpu().numpy(), boundaries.cpu().numpy(), centroids.cpu().numpy(), nbits)
                assert (result.cpu().numpy().view(np.uint32) == res_o.view(np.uint32)).all(), (shift, k)
                assert (packed.cpu().numpy().view(np.uint32) == oracle.bins_to_bits(bins_o, nbits)).all(), (shift, k)
            for size in (0, 1 << 13, 1 << 15, 1 << 18, 1 << 20, 1 << 22):
                vec = torch.cat([others[:size], x])
                slices = [(0, size, size, 1)] * (size > 0) + [(size, n, n, 1)]
                got, scale = capi.host().eden_compress(vec, boundaries, centroids, nbits, seed, slices)[-1]
                assert torch.equal(scale.view(torch.int32), result[2].view(torch.int32)), (shift, k, size)
                assert torch.equal(got, packed), (shift, k, size)


@pytest.mark.parametrize("seed", [2 ** 63 + 5, -(2 ** 63), 2 ** 70 + 9, 2 ** 64 - 1])
def test_seeds_of_any_size(capi, seed):
    """a seed is taken modulo 2^64, as the single calls take it; one that is no whole number is refused"""
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    eden = Eden(device=DEV)
    x = torch.randn(3000, device=DEV)
    data = eden.compress(x, 4, seed)
    low = (seed + 2 ** 63) % 2 ** 64 - 2 ** 63
    want = eden.compress(x, 4, low)
    assert all(torch.equal(a["packed_bins"], b["packed_bins"]) and a["seed"] == seed for a, b in zip(data, want))
    assert torch.equal(eden.decompress(data), eden.decompress(want))
    with pytest.raises(TypeError):
        eden.compress(x, 4, 1.0)


def test_handles_and_seeds_that_int_takes(capi):
    """streams as handles of numpy's types, seeds and steps as floats: whatever int() makes a whole number of"""
    import math
    n, side = 1 << 14, torch.cuda.Stream()
    x = torch.randn(n, device=DEV)
    size = capi.required_bytes(n, 4, 16, 2)
    a, b = torch.zeros(size, dtype=torch.uint8, device=DEV), torch.zeros(size, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    capi.rht_scaling_compress(x, None, a, 1024, 1 / math.sqrt(1024), 4, 2, seed=7, step=2 ** 64 + 3, stream=side)
    capi.rht_scaling_compress(x, None, b, 1024, 1 / math.sqrt(1024), 4, 2, seed=np.float64(7), step=3.0, stream=np.int64(side.cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(a, b) and int(a.sum()) > 0


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("nbits", [1, 8])
@pytest.mark.parametrize("sizes", [[(32, 1), (32, 3), (512, 2), (1024, 0), (4096, 1), (8192, 2), (8192, 1), (256, 1), (2048, 1), (64, 2)],
                                   [(16384, 1)] * 9 + [(1 << 15, 1), (1 << 17, 1), (16384, 2), (16384, 0), (1 << 16, 3)],
                                   [(16384, 1), (16384, 2), (8192, 1), (16384, 0), (1 << 15, 2)],
                                   [(1 << 22, 1), (1 << 14, 1), (1 << 13, 1), (1 << 23, 1), (1 << 18, 2)]])
def test_many_slices_share_launches(capi, sizes, nbits, dt):
    """slices of every kind in one call -- more than a launch takes, one workgroup each, passes shared, by themselves, with no, one
    and several rotations, ragged -- against the calls they stand for"""
    import math
    from dynamiq_sigcomm_artifact_amd.eden import Eden
    eden, host, seed = Eden(device=DEV), capi.host(), -3
    centroids, boundaries = eden._tables(nbits)
    slices, start = [], 0
    for k, (size, rotations) in enumerate(sizes):
        count = size - (k % 3) * (size // 40 + 1)
        slices.append((start, count, size, rotations))
        start += count
    g = torch.Generator(device=DEV).manual_seed(nbits)
    vec = (torch.randn(start, generator=g, device=DEV) * 1e-2).to(dt)
    got = host.eden_compress(vec, boundaries, centroids, nbits, seed, slices)
    want = []
    for (packed, scale), (at, count, size, rotations) in zip(got, slices):
        inv = float(np.float32(1.0) / np.float32(math.sqrt(size)))
        x = torch.zeros(size, device=DEV)
        x[:count] = vec[at:at + count].float()
        diags = [torch.empty(size, device=DEV) for _ in range(rotations)]
        for i, diag in enumerate(diags):
            capi.rand_diag(diag, seed + i)
            capi.rht_blocked(x, diag, size, inv, False)
        ref, result = torch.empty_like(packed), torch.empty(4, device=DEV)
        capi.eden_quantize(x, boundaries, centroids, nbits, ref, result, torch.empty(capi.eden_work_doubles(size), dtype=torch.float64, device=DEV))
        assert torch.equal(packed, ref) and torch.equal(scale.view(torch.int32), result[2].view(torch.int32)), (count, size, rotations)
        y = torch.empty(size, device=DEV)
        capi.eden_dequantize(ref, size, centroids, nbits, y)
        for diag in reversed(diags):
            capi.rht_blocked(y, diag, size, inv, True)
        want.append((result[2] * y)[:count].to(dt))
    out = torch.empty(start, dtype=dt, device=DEV)
    host.eden_decompress(out, [(p, nbits, centroids, s, count, rotations, seed) for (p, s), (_, count, _, rotations) in zip(got, slices)])
    assert torch.equal(out, torch.cat(want))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [16385, 20255, 1 << 15])
def test_thc_of_one_block_of_2p15_is_that_of_a_long_vector(capi, n, dt):
    """THC's compress and decompress of one block of 2^15 in two passes, with a source and a destination shorter than the block and the grid
    from a norm on the device, against the first of 40 blocks, which take one pass, with the quantisers on their own"""
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    dim, name = 1 << 15, (0, 1)
    c = OldINCACudaHadamardCompressor({"d": {name: dim}, "size": {name: n}, "T": 2.7, "device": DEV, "nclients": 6, "rank": 0})
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(n, generator=g, device=DEV).to(dt)
    norm, u = x.float().norm(), torch.rand(dim, generator=g, device=DEV)
    levels = c.compress(x, name, norm, uniform=u)
    rot = c.hadamards[name]
    low, spacing = c._grid(norm, dim)
    signs = torch.cat([rot.diagonal_bits] * 40)
    long = torch.zeros(40 * dim, device=DEV)
    long[:n] = x.float()
    capi.rht_blocked(long, signs, dim, rot.inv_sqrt, False)
    want = torch.empty(dim, dtype=torch.bfloat16, device=DEV)
    capi.thc_quantize(long[:dim].contiguous(), u, want, low.reshape(1), spacing.reshape(1), 64)
    assert torch.equal(levels.view(torch.int16), want.view(torch.int16)) and want.unique().numel() > 32
    total = (levels.float() * 6).to(torch.bfloat16)
    got = c.decompress(total, name).clone()
    back = torch.empty(dim, device=DEV)
    capi.thc_dequantize(total, back, (spacing / 6).reshape(1), low.reshape(1))
    long.zero_()
    long[:dim] = back
    capi.rht_blocked(long, signs, dim, rot.inv_sqrt, True)
    assert got.numel() == n and torch.equal(got.view(torch.int32), long[:n].view(torch.int32))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,dim", [(1024, 1024), (40000, 65536), (1 << 20, 1 << 20), (1000, 1024), ((1 << 21) + 5, 1 << 22),
                                   (20255, 1 << 15), (16385, 1 << 15), (1 << 15, 1 << 15)])
def test_thc_grid_and_source_in_the_passes(capi, n, dim, dt):
    """THC's compress and decompress with the grid from a norm on the device, from a number, and as torch works it out
    (a norm of another type takes the single calls); sources of another type, length and alignment than the transform"""
    from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor
    dev = "cuda:0"
    c = OldINCACudaHadamardCompressor({"d": {(0, 1): dim}, "size": {(0, 1): n}, "T": 2.7, "device": dev, "nclients": 6, "rank": 0})
    g = torch.Generator(device=dev).manual_seed(dim)
    x = torch.randn(n + 1, generator=g, device=dev).to(dt)[n & 1:][:n]
    norm = x.float().norm()
    u = torch.rand(dim, generator=g, device=dev)
    name = (0, 1)
    levels = c.compress(x, name, norm, uniform=u)
    work = torch.zeros(dim, device=dev)
    work[:n] = x.float()
    low, spacing = c._grid(norm, dim)
    want = torch.empty(dim, dtype=torch.bfloat16, device=dev)
    rot = c.hadamards[name]
    capi.thc_rht_quantize(work, rot.diagonal_bits, u, want, dim, rot.inv_sqrt, low.reshape(1), spacing.reshape(1), 64)
    assert torch.equal(levels, want)
    total = (levels.float() * 6).to(torch.bfloat16)
    got = c.decompress(total, name).clone()
    back = torch.empty(dim, device=dev)
    capi.thc_dequantize_irht(total, rot.diagonal_bits, back, dim, rot.inv_sqrt, (spacing / 6).reshape(1), low.reshape(1))
    assert got.numel() == n and torch.equal(got, back[:n])
    host = c.compress(x, name, float(norm), uniform=u)                         # the grid from a number: rounded once
    assert (host.float() - want.float()).abs().max() <= 1 and (host != want).float().mean() < 1e-3
    assert (c.decompress(total, name) - got).norm() < 1e-5 * got.norm()
    double = c.compress(x, name, norm.double(), uniform=u)
    assert (double != host).float().mean() < 1e-3
